"""The reciprocal, root and quotient steps of the shading and the adjoint
(polyred_amd/csrc/roots.hpp) on the MI355X: correctly rounded for every float32
mantissa at every exponent of their ranges (quotients: for every divisor's
mantissa, over mixed numerators and the ones nearest a rounding boundary).  The
frames' bit-exactness rests on this hardware's estimates there."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    so = os.path.join(HERE, "_build", "libroots.so")
    if not os.path.exists(so):
        subprocess.run(["make", "-s", "-C", HERE], check=True)
    L = C.CDLL(so)
    L.roots_check.argtypes = [C.c_int, C.c_int, C.c_int, C.POINTER(C.c_ulonglong), C.POINTER(C.c_uint32)]
    return L


def _run(lib, which, a, b):
    n, one = C.c_ulonglong(), (C.c_uint32 * 2)()
    assert lib.roots_check(which, a, b, C.byref(n), one) == 0
    assert n.value == 0, (n.value, hex(one[0]), hex(one[1]))


def test_reciprocals(lib, device):
    _run(lib, 0, -100, 100)


def test_roots(lib, device):
    _run(lib, 1, -64, 64)


@pytest.mark.parametrize("seed", [1, 2])
def test_quotients(lib, device, seed):
    _run(lib, 2, 64, seed)
