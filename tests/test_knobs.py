"""What a frame makes of a renderer's speed knobs (knobs.hpp, built for the
host): the rules on the frame's size decide for a knob nobody set, and a knob
a caller set is taken at its value, the default's too."""
import ctypes as C
import os
import subprocess

import pytest

from polyred_amd import abi

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "polyred_amd", "csrc")

SRC = r'''
#include "knobs.hpp"
using namespace prh;
// the knobs of a new renderer, or of one that `t` was set on: the setup's
// threshold, in the low bits, and whether the frame takes two streams
extern "C" int frame(const prh_tuning* t, long pixels, long n_tris, int ao, int wide) {
    Knobs k = default_knobs((size_t)pixels);
    if (t) set_knobs(k, *t);
    return direct_centres(k, n_tris, wide) | (two_streams(k, (size_t)pixels, n_tris, ao) ? 1024 : 0);
}
extern "C" void defaults(long pixels, prh_tuning* t) { *t = default_knobs((size_t)pixels); }
extern "C" int valid(const prh_tuning* t) { return valid_knobs(*t); }
'''


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("knobs")
    src, so = d / "k.cpp", d / "k.so"
    src.write_text(SRC)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(src), "-o", str(so)], check=True)
    L = C.CDLL(str(so))
    L.frame.argtypes = [C.POINTER(abi.prh_tuning), C.c_long, C.c_long, C.c_int, C.c_int]
    L.defaults.argtypes = [C.c_long, C.POINTER(abi.prh_tuning)]
    L.valid.argtypes = [C.POINTER(abi.prh_tuning)]
    return L


SIZES = [(480 * 270, 197_000), (1001 * 701, 310_000), (1920 * 1080, 1 << 19), (1920 * 1080, (1 << 19) + 1),
         (3840 * 2160, 116_000), (3840 * 2160, 1_040_000), (1 << 19, 10), ((1 << 19) - 1, 10), (1, 0)]


@pytest.mark.parametrize("pixels,tris", SIZES)
@pytest.mark.parametrize("ao", [0, 1])
def test_set_knobs_are_taken(lib, pixels, tris, ao):
    t = abi.prh_tuning()
    lib.defaults(pixels, C.byref(t))
    for direct in (0, 16, 24, 47, 48, 49, 256):
        for overlap in (0, 1):
            for wide in (0, 1):
                t.main_direct_max, t.overlap_shadows = direct, overlap
                assert lib.valid(C.byref(t))
                assert lib.frame(C.byref(t), pixels, tris, ao, wide) == direct + 1024 * overlap


@pytest.mark.parametrize("pixels,tris", SIZES)
@pytest.mark.parametrize("ao", [0, 1])
def test_rules_of_unset_knobs(lib, pixels, tris, ao):
    t = abi.prh_tuning()
    lib.defaults(pixels, C.byref(t))
    assert (t.raster_wg_per_cu, t.item_prims, t.shadow_direct_max, t.main_direct_max, t.raster_tile) == (8, 2048, 64, 48, 16)
    assert t.overlap_shadows == (pixels >= 1 << 19)
    two = pixels >= 1 << 19 and (tris > 1 << 19 or (ao and pixels >= 1 << 22))
    assert lib.frame(None, pixels, tris, ao, 0) == (16 if tris <= 1 << 19 else 48) + 1024 * two
    assert lib.frame(None, pixels, tris, ao, 1) & 1023 == 48


def test_refusals(lib):
    for bad in (dict(item_prims=1000), dict(item_prims=32), dict(item_prims=0), dict(item_prims=16384),
                dict(raster_wg_per_cu=0), dict(raster_wg_per_cu=17), dict(main_direct_max=-1), dict(main_direct_max=257),
                dict(shadow_direct_max=-1), dict(shadow_direct_max=257), dict(overlap_shadows=2),
                dict(overlap_shadows=-1), dict(raster_tile=0), dict(raster_tile=24), dict(raster_tile=64)):
        t = abi.prh_tuning()
        lib.defaults(1 << 20, C.byref(t))
        for k, v in bad.items():
            setattr(t, k, v)
        assert not lib.valid(C.byref(t)), bad
