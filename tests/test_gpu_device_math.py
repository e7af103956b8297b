"""The kernels' short arithmetic against the compiler's own, to the last bit, over
every argument it takes: the reciprocal root of all 2^32 floats, the two divisors
of the packed normals and tangents over all whole numbers of 16 bits."""

import ctypes
import os

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", [0, 32767, 16383], ids=["reciprocal root", "divide by 32767", "divide by 16383"])
def test_short_forms_have_the_same_bits(which):
    lib = ctypes.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libdevice_math.so"))
    lib.device_math_differences.restype = ctypes.c_longlong
    assert lib.device_math_differences(which) == 0
