"""The AO's angle and power without the library functions (gomath.hpp, built
for the host): float32(atan(r)) for 0 < r <= 2^-5 against the C library's for
every float32 from 2^-13 up and for samples below (where it is r), and
pow32_fast at the exponent 10000 for every float32 base of the last binades
below 1 whose power does not vanish."""
import ctypes as C
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "polyred_amd", "csrc")

SRC = r'''
#include <cmath>
#include <cstring>
#include "gomath.hpp"
static float of(unsigned u) { float f; std::memcpy(&f, &u, 4); return f; }
static unsigned bits(float f) { unsigned u; std::memcpy(&u, &f, 4); return u; }
// the first float32 of the bit range that differs (0: none)
extern "C" unsigned atan_first_bad(unsigned lo, unsigned hi, unsigned step) {
    for (unsigned u = lo; u <= hi; u += step)
        if (bits(gm::atan32_small(of(u))) != bits((float)std::atan((double)of(u)))) return u;
    return 0;
}
extern "C" unsigned pow_first_bad(unsigned lo, unsigned hi, unsigned step) {
    for (unsigned u = lo; u <= hi; u += step)
        if (bits(gm::pow32_fast(of(u), 10000.0f)) != bits((float)std::pow((double)of(u), 10000.0))) return u;
    return 0;
}
'''


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("aomath")
    src, so = d / "p.cpp", d / "p.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-mfma", "-std=c++17", "-ffp-contract=off", "-fPIC", "-shared", f"-I{CSRC}", str(src),
                    "-o", str(so)], check=True)
    L = C.CDLL(str(so))
    for f in (L.atan_first_bad, L.pow_first_bad):
        f.argtypes, f.restype = [C.c_uint] * 3, C.c_uint
    return L


def b(x):
    import struct
    return struct.unpack("<I", struct.pack("<f", x))[0]


def test_atan(lib):
    assert lib.atan_first_bad(b(2.0 ** -13), b(2.0 ** -5), 1) == 0
    assert lib.atan_first_bad(b(2.0 ** -149), b(2.0 ** -13), 1009) == 0


def test_power(lib):
    # 0.9894^10000 is below 2^-150, the smallest that rounds up from zero
    assert lib.pow_first_bad(b(0.9893), b(1.0), 1) == 0
    assert lib.pow_first_bad(b(2.0 ** -20), b(0.9893), 4099) == 0
