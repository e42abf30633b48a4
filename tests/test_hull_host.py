"""The cascade lane compiled for the host: the hull test that lets a sub-step pass without the exact comparator must
agree with it, at the very edge of the test's margin, whatever the stages' time constants (far apart ones make terms of
1e5 and more that cancel)."""
import pathlib
import re
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent
SENSOR = HERE.parent / "ballasim_amd" / "csrc" / "sensor"


@pytest.fixture(scope="module")
def hull_check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("hull_check") / "hull_check"
    subprocess.run(["g++", "-O2", "-std=c++20", "-ffp-contract=off", f"-I{SENSOR}", "-o", str(exe),
                    str(HERE / "host" / "hull_check.cpp")], check=True)
    return exe


@pytest.mark.parametrize("ratio", ["10", "1e3", "1e5", "1e6", "1e7"])
def test_hull_passes_no_crossing(hull_check, ratio):
    for seed in (1, 2):
        r = subprocess.run([str(hull_check), "500", str(seed), ratio], capture_output=True, text=True, timeout=110)
        assert r.returncode == 0, r.stdout
        quick, near, bad = map(int, re.search(r"quick (\d+) near (\d+) crossings (\d+)", r.stdout).groups())
        assert bad == 0
        assert quick > 100000 and near > 50000  # passes, and passes at the margin's edge
