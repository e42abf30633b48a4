"""The helper that spreads a call's work over threads (csrc/core/workers.h), on the host: when allocations fail while
the threads are being started, whichever it is, every piece of work is still done once and the call returns."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent
CORE = HERE.parent / "ballasim_amd" / "csrc" / "core"


@pytest.fixture(scope="module")
def workers_check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("workers") / "workers_check"
    subprocess.run(["g++", "-O2", "-std=c++20", "-pthread", f"-I{CORE}", "-o", str(exe),
                    str(HERE / "host" / "workers_check.cpp")], check=True)
    return exe


def test_every_piece_is_done_once(workers_check):
    assert subprocess.run([str(workers_check)]).returncode == 0


@pytest.mark.parametrize("failures", [1, 1000])
@pytest.mark.parametrize("first", range(16))
def test_no_memory_for_threads(workers_check, first, failures):
    r = subprocess.run([str(workers_check), str(first), str(failures)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
