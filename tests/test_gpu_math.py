"""The device math the exact searches rely on (GPU): pm::log is monotone on every positive float
and equals the oracle's log bit for bit (an order-independent hash of all 2^31 - 2^23 results
against the one the oracle produced, recorded in the golden manifest). And the device's forms of the
fp32 functions, which divide by reciprocal and remainder, give the bits of the host's plain divisions."""
import ctypes as C
import json
import os
import pathlib
import shutil
import subprocess

import numpy as np
import pytest

from ballasim_amd import _abi

pytestmark = pytest.mark.gpu


def test_device_log_monotone_and_equal_to_oracle():
    lib = _abi.load_library()
    v, h = C.c_uint64(0), C.c_uint64(1)
    _abi.check(lib.bsx_math_selfcheck(C.byref(v), C.byref(h)))
    man = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "manifest.json")))["log_check"]
    assert v.value == 0
    assert "0x%016x" % h.value == man["hash"]


def _bits(x):
    return int(np.float32(x).view(np.uint32))


# (function, first, last): the whole range its callers can reach, as bit patterns (13: div_with on drawn pairs)
MATH = [(0, 0, 0x7fffffff), (1, 0, 0xffffffff), (2, 0, 0x7fffffff), (3, 0, 0xffffffff)] + \
       [(f, 0, _bits(1e12)) for f in (4, 5, 6, 7)] + \
       [(f, _bits(2.0 ** -100), _bits(2.0 ** 100)) for f in (8, 9, 10, 11)] + \
       [(f, 0x7f7fffff, 0x7fc00001) for f in (9, 10)] + \
       [(12, _bits(2.0 ** -120), _bits(2.0 ** 120)), (13, 0, 0xffffffff)]


@pytest.fixture(scope="module")
def host_hash(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    here = pathlib.Path(__file__).resolve().parent
    exe = tmp_path_factory.mktemp("math") / "math_hash"
    subprocess.run(["g++", "-O3", "-march=native", "-std=c++17", "-ffp-contract=off", "-pthread",
                    f"-I{here.parent / 'ballasim_amd' / 'csrc' / 'core'}", "-o", str(exe),
                    str(here / "host" / "math_hash.cpp")], check=True)
    return exe


@pytest.mark.parametrize("fn,first,last", MATH)
def test_device_functions_equal_plain_division(host_hash, fn, first, last):
    """Every bit pattern of the range (of the pairs of div_with, one drawn from each of the 2^32)."""
    h = C.c_uint64(0)
    _abi.check(_abi.load_library().bsx_math_hash(fn, first, last, 1, C.byref(h)))
    r = subprocess.run([str(host_hash), str(fn), str(first), str(last), "1"], capture_output=True, text=True, check=True)
    assert h.value == int(r.stdout)
