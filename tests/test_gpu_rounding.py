"""The surface searches' bits rest on recip_rn and sqrt_rn (csrc/vsdmo_numerics.h)
being correctly rounded, which one step from the hardware's approximations is
not by itself: every value of their ranges against 1.0f / x and sqrtf(x)."""
import ctypes as C
import os
import subprocess

import pytest

from volumesurfacediscretemeshoptimization_amd import build

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "hip", "rounding.so")


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        subprocess.run([build.hipcc(), *build.HIPCC_FLAGS, "-I", build.CSRC, "-o", LIB,
                        os.path.join(HERE, "hip", "rounding.hip")], check=True, timeout=100)
    lib = C.CDLL(LIB)
    lib.rounding_compare.argtypes = [C.c_int, C.c_uint, C.c_uint, C.POINTER(C.c_ulonglong)]
    return lib


# biased exponents: recip_rn [2^-126, 2^126), sqrt_rn [2^-96, 2^128)
@pytest.mark.parametrize("root,lo,hi", [(0, 1, 64), (0, 64, 128), (0, 128, 192), (0, 192, 253),
                                        (1, 31, 96), (1, 96, 160), (1, 160, 255)])
def test_every_value(lib, root, lo, hi):
    out = (C.c_ulonglong * 2)()
    assert lib.rounding_compare(root, lo, hi, out) == 0
    assert out[1] == (hi - lo) << 23
    assert out[0] == 0, f"{out[0]} of {out[1]} values differ"
