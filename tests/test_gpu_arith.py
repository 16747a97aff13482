"""The fast arithmetic of the RK5 kernels on the device (step factors from the
hardware's log2 and exp2, division by a double reciprocal, the exponential
without its clamps) gives the bits of the forms it replaces, for every float
of its range (tests/device/arith_check.hip, built with the library)."""
import ctypes
import os

import numpy as np
import pytest

from conftest import ROOT, gpu_available

pytestmark = pytest.mark.gpu

POW_FAST, POW_CHAIN, DIV_RECIP, DIV_EPS, EXP_NEAR, DIV_PAIRS = range(6)
ALL = 1 << 32


@pytest.fixture(scope="module")
def check():
    if not gpu_available():
        pytest.skip("no GPU")
    lib = ctypes.CDLL(os.path.join(ROOT, "tests", "device", "libarith_check.so"))
    lib.arith_check.restype = ctypes.c_longlong
    lib.arith_check.argtypes = [ctypes.c_int, ctypes.c_float, ctypes.c_ulonglong, ctypes.c_ulonglong]
    return lib.arith_check


def test_every_pattern_is_visited(check):
    assert check(-1, 1.0, 0, ALL) == ALL and check(-1, 1.0, 5, 1005) == 1000


@pytest.mark.parametrize("what", [POW_FAST, POW_CHAIN, DIV_EPS, EXP_NEAR])
def test_every_float(check, what):
    assert check(what, 1.0, 0, ALL) == 0


# time constants and capacitances, powers of two, significands that stress the
# rounding (1 + ulp, all ones, pi) and the ends of the normal range
@pytest.mark.parametrize("bits", [0x438C8000, 0x43100000, 0x41A00000, 0x3DCCCCCD, 0x358637BD,
                                  0x40400000, 0xC0E00000, 0x3F800000, 0x40000000, 0x3F800001,
                                  0x3FFFFFFF, 0x40490FDB, 0x00800000, 0x00FFFFFF, 0x7E800000,
                                  0x7F7FFFFF])
def test_division_of_every_float(check, bits):
    d = float(np.array([bits], np.uint32).view(np.float32)[0])
    assert check(DIV_RECIP, d, 0, ALL) == 0


def test_division_of_pairs(check):
    # 2^32 pairs over all dividends and all normal divisors
    assert check(DIV_PAIRS, 1.0, 0, ALL) == 0
