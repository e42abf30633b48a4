"""The memory rule of the cascade's segment coefficients (csrc/sensor/coefs.h) over recordings whose windows grow: the
buffer grows a few times and not with every window, up to a quarter of the memory that is free without it, and a window
within that share is served whatever the buffer holds already."""
import pathlib
import re
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent
SENSOR = HERE.parent / "ballasim_amd" / "csrc" / "sensor"


@pytest.fixture(scope="module")
def coefs_check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("coefs") / "coefs_check"
    subprocess.run(["g++", "-O2", "-std=c++20", f"-I{SENSOR}", "-o", str(exe), str(HERE / "host" / "coefs_check.cpp")],
                   check=True)
    return exe


def _run(exe, windows, need, per_mille, device):
    r = subprocess.run([str(exe), str(windows), str(need), str(per_mille), str(device)], capture_output=True, text=True)
    assert r.returncode == 0
    grown, without, share = re.search(r"grown (\d+) without (\d+) share ([0-9.]+)", r.stdout).groups()
    return int(grown), int(without), float(share)


def test_windows_that_grow_a_little_do_not_each_reallocate(coefs_check):
    grown, without, share = _run(coefs_check, 100, 1e9, 10, 288e9)  # 1 GB to 2.7 GB, 1 % a window
    assert without == 0 and grown <= 6, grown


def test_the_held_buffer_counts_as_free(coefs_check):
    # from 15 % to 24 % of the device: each within a quarter of what is free without the buffer
    grown, without, share = _run(coefs_check, 48, 6e9, 10, 40e9)
    assert without == 0 and share <= 0.25, (without, share)


def test_never_past_its_share(coefs_check):
    grown, without, share = _run(coefs_check, 60, 6e9, 50, 40e9)
    assert without > 0 and share <= 0.25
    grown, without, share = _run(coefs_check, 60, 20e9, 20, 288e9)  # (or 32 GiB)
    assert without > 0 and share * 288e9 <= 32 * 2 ** 30 + 1e6
