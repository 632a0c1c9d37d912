"""The differentiable shading at a shininess of 0 (a model material without
Ns; also the lower bound a fit keeps it at) on the MI355X through the C ABI.
x^0 is 1 for every cosine, and its derivative by the exponent, x^s log x, is
taken where 0 < x < 1 only: a light behind a pixel's half vector (x = 0) adds
nothing.  Against the FP64 reference, whose rule that is, at test_gpu_diff's
bars; and a fit that starts at 0 or is driven there stays finite."""
import numpy as np
import pytest

import oracle
from polyred_amd import abi, diff, render, scenes

from .test_gpu_adjoint_sizes import _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_lights", [4, 8])
@pytest.mark.parametrize("zero", [(0,), (1, 4), tuple(range(8))])
def test_backward(device, orc, n_lights, zero):
    s = _scene(96, 80, n_lights=n_lights)
    r = render.renderer_for(s, device)
    r.render_device()
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    p = diff.scene_params(s)
    p.shininess[list(zero)] = 0.0
    lin = r.ForwardLinear(p)
    target = np.nan_to_num(0.5 * lin).astype(np.float32)
    ref_loss, _, gref = oracle.diff(s, order, p, target.astype(np.float64))
    for noalloc in (False, True):
        loss, g = diff.backward(r._lib, r.handle, p, target, s.height, s.width, noalloc=noalloc)
        assert abs(loss - ref_loss) <= 1e-4 * ref_loss, (loss, ref_loss)
        for n in diff.DiffParams.NAMES:
            a = np.asarray(getattr(g, n), np.float64).reshape(-1)
            b = np.asarray(gref[n], np.float64).reshape(-1)
            assert np.isfinite(a).all(), n
            assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b) + 1e-12, n
    r.free()


@pytest.mark.parametrize("stored", [False, True])
def test_fit(device, stored):
    s, views = scenes.c5_inverse(seed=23, n_views=2, n_spheres=9, min_side=60, max_side=90, shadow_size=128)
    gs, rs = render.views_of(s, views, device)
    for r in rs:
        r.render_device()
    truth = diff.scene_params(s)
    start = truth.copy()
    start.shininess[0] = 0.0   # p = 0 (1 + theta): stays
    start.shininess[1] = 30.0  # above the truth: the first step, -2 in theta, meets the bound
    truth.shininess[1] = 1.0
    fit = diff.Fit(rs, stored_gbuffer=stored)
    fit.targets(truth)
    p, _ = fit.run(start, steps=1, lr=2.0, groups=("shininess",))
    assert p.shininess[1] == 0.0
    p, hist = fit.run(start, steps=4, lr=2.0, groups=("shininess",))
    assert np.isfinite(hist).all()
    assert p.shininess[0] == 0.0
    assert np.isfinite(p.shininess).all() and (p.shininess >= 0).all()
    # and every other group beside it
    q, hist = fit.run(start, steps=4, lr=1e-2)
    assert np.isfinite(hist).all()
    for n in ("kd", "ks", "shininess", "light_pos", "light_int"):
        assert np.isfinite(getattr(q, n)).all(), n
    fit.free()
    gs.free()
