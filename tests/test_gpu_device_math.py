"""GPU check of the short square roots and quotients (tests/device_math.hip): from
the device's own starting values the reciprocal, the square root and its inverse
are correctly rounded for every mantissa, at exponents of both parities across the
range they are used in."""
import ctypes
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "libdevice_math.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        subprocess.run(["make", "-C", HERE], check=True)
    so = ctypes.CDLL(LIB)
    so.device_math_wrong.restype = ctypes.c_long
    so.device_math_wrong.argtypes = [ctypes.c_uint32]
    return so


@pytest.mark.parametrize("exponent", [32, 87, 126, 127, 128, 167, 222])
def test_every_mantissa(lib, exponent):
    print(f"case device math exponent={exponent}", flush=True)
    assert lib.device_math_wrong(exponent) == 0
