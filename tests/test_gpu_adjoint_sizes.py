"""The adjoint's list of shaded pixels and its light variants at the sizes
where they can go wrong, on the MI355X through the C ABI against the FP64
reference (oracle_diff): images of one pixel, of one row or column, around
the 8x8 blocks, 16x16 tiles and 64-pixel strips and chunks of the list; 0, 1,
4, 5 and 8 lights (the kernels hold up to 4 or up to 8), point and
directional; flat and smooth shading; a material table past the LDS bins.

The target is half of the forward at the same parameters, so that neither the
residual nor the sums cancel: each is then float32 arithmetic of relative
error a few 1e-6 a pixel, and 1e-3 of a group's norm (the bar of
test_gpu_diff) is far above it."""
import numpy as np
import pytest

import oracle
from polyred_amd import abi, diff, render, scenes

pytestmark = pytest.mark.gpu


def _scene(w, h, n_lights=4, flat=False, n_mats=8):
    s = scenes.c4_adjoint(seed=31, width=w, height=h, n_spheres=40)
    # a wide aspect ratio keeps the objects in view; every fourth pixel or so is empty
    s.camera = dict(s.camera, position=(0.0, 1.0, 13.0))
    proto = s.lights
    s.lights = []
    for i in range(n_lights):
        l = proto[i % len(proto)]
        if i % 3 == 2:
            s.lights.append(scenes.Light(kind=abi.PRH_LIGHT_DIRECTIONAL, direction=scenes.unit3((0.1 * i, -1.0, -0.4)),
                                         intensity=0.6, color=l.color))
        else:
            s.lights.append(scenes.Light(position=tuple(float(np.float32(c + i)) for c in l.position), intensity=4.0,
                                         color=l.color))
    proto = s.materials
    s.materials = [scenes.Material(**vars(proto[i % len(proto)])) for i in range(n_mats)]
    for i, m in enumerate(s.materials):
        m.flat_shading = flat and i % 2 == 0
    s.obj_mat_base = (np.arange(len(s.obj_mat_base)) * 7) % n_mats
    return s


def _check(device, s):
    r = render.renderer_for(s, device)
    r.render_device()
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    p = diff.scene_params(s)
    lin = r.ForwardLinear(p)
    _, ref, _ = oracle.diff(s, order, p)
    shaded = ~np.isnan(ref).any(-1)
    assert np.array_equal(shaded, ~np.isnan(lin).any(-1))
    target = np.nan_to_num(0.5 * lin).astype(np.float32)
    for noalloc in (False, True):
        loss, g = diff.backward(r._lib, r.handle, p, target, s.height, s.width, noalloc=noalloc)
        if not shaded.any():
            assert loss == 0 and all(not getattr(g, n).any() for n in diff.DiffParams.NAMES)
            continue
        ref_loss, _, gref = oracle.diff(s, order, p, target.astype(np.float64))
        assert abs(loss - ref_loss) <= 1e-4 * ref_loss, (loss, ref_loss)
        for n in diff.DiffParams.NAMES:
            a = np.asarray(getattr(g, n), np.float64).reshape(-1)
            b = np.asarray(gref[n], np.float64).reshape(-1)
            assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b) + 1e-12, (n, np.linalg.norm(a - b), np.linalg.norm(b))
    r.free()
    return int(shaded.sum())


@pytest.mark.parametrize("w,h", [(1, 1), (1, 40), (40, 1), (7, 9), (8, 8), (16, 16), (17, 15), (63, 17), (64, 64), (65, 33),
                                 (129, 50), (200, 131)])
def test_any_image_size(device, orc, w, h):
    n = _check(device, _scene(w, h))
    assert n > 0 or w * h <= 64


@pytest.mark.parametrize("n_lights", [0, 1, 4, 5, 8])
@pytest.mark.parametrize("flat", [False, True])
def test_any_light_count(device, orc, n_lights, flat):
    assert _check(device, _scene(90, 70, n_lights=n_lights, flat=flat)) > 1000


# 4096 LDS slots hold 7 values of up to 18 materials in 32 copies, ..., of up
# to 585 in one; past that, and past 512 the gradients have no replicas
@pytest.mark.parametrize("n_mats", [1, 18, 19, 36, 37, 292, 293, 512, 513, 585, 586, 700])
def test_any_material_count(device, orc, n_mats):
    assert _check(device, _scene(90, 70, n_mats=n_mats)) > 1000
