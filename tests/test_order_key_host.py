"""The output stage's sort key on the host (csrc/output/order_key.h): one integer in the order of (t_reported, x, y,
t_cross), whatever the readout, and buckets by its leading bits that one block each can sort, also where the readout's
quantum leaves a window few reported times."""
import pathlib
import re
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent
CSRC = HERE.parent / "ballasim_amd" / "csrc"


@pytest.fixture(scope="module")
def order_key_check(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("order_key") / "order_key_check"
    subprocess.run(["g++", "-O2", "-std=c++20", "-ffp-contract=off", f"-I{CSRC / 'output'}", "-o", str(exe),
                    str(HERE / "host" / "order_key_check.cpp")], check=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2])
def test_keys_have_the_output_order(order_key_check, seed):
    r = subprocess.run([str(order_key_check), "order", "6000", str(seed)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout
    used, shifted, wide, bad = map(int, re.search(r"trials (\d+) shifted (\d+) wide (\d+) differences (\d+)",
                                                  r.stdout).groups())
    assert bad == 0 and used > 3000
    assert shifted > used // 4  # quanta that the key divides out are exercised


@pytest.mark.parametrize("quantum_ns", [0, 1000, 6000, 20000, 100000, 10 ** 6, 5 * 10 ** 6, 10 ** 8])
@pytest.mark.parametrize("n,size,drift", [(2900000, (2048, 1536), 0.0), (900000, (1280, 720), 35.0),
                                          (30000, (640, 480), -4000.0)])
def test_buckets_fit_a_block_at_any_quantum(order_key_check, n, size, drift, quantum_ns):
    r = subprocess.run([str(order_key_check), "fill", str(n), str(size[0]), str(size[1]), str(quantum_ns), str(drift)],
                       capture_output=True, text=True, timeout=120)
    largest, cap = map(int, re.search(r"largest (\d+) cap (\d+)", r.stdout).groups())
    assert largest <= cap, r.stdout


# Where even events spread evenly are too many for blocks to sort, the bucket passes are not tried; below, they are.
@pytest.mark.parametrize("n,size,quantum_ns,tried", [(2049, (3, 2), 0, True), (8000000, (2048, 1536), 1000, True),
                                                     (20000000, (2048, 1536), 1000, False)])
def test_bucket_passes_are_not_tried_in_vain(order_key_check, n, size, quantum_ns, tried):
    r = subprocess.run([str(order_key_check), "fill", str(n), str(size[0]), str(size[1]), str(quantum_ns), "0"],
                       capture_output=True, text=True, timeout=120)
    assert ("too many" not in r.stdout) == tried, r.stdout
