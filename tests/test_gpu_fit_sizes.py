"""The fit's update over parameter counts around the kernels' own sizes
(256 parameters a workgroup of the Adam pass, and the material counts at
which the adjoint's accumulation changes), on the MI355X through the C ABI:
two steps against a float64 Adam on the host fed the single-view gradients
at each step's parameters, so that a gradient, loss or step counter left
over from the first step would show in the second."""
import numpy as np
import pytest

from polyred_amd import diff, render, scenes

from .test_gpu_fit import _adam64, _summed_backward

pytestmark = pytest.mark.gpu


# 3 kd values a material: 255, 258, 513 and 1536 parameters without the
# vertex colours; 1, 8 materials; 300 and 512 exceed 256 materials
@pytest.mark.parametrize("n_mats", [1, 8, 31, 33, 85, 86, 171, 300, 512])
@pytest.mark.parametrize("groups", [("kd",), ("kd", "albedo", "ks", "shininess", "light_pos", "light_int")])
def test_two_steps_any_material_count(device, n_mats, groups):
    s, views = scenes.c5_inverse(seed=21, n_views=2, n_spheres=9, min_side=60, max_side=90, shadow_size=128)
    proto = s.materials
    s.materials = [proto[i % len(proto)] for i in range(n_mats)]
    s.obj_mat_base = (np.arange(len(s.obj_mat_base)) * 37) % n_mats
    gs, rs = render.views_of(s, views, device)
    for r in rs:
        r.render_device()
    p0 = diff.scene_params(s)
    truth = diff.perturb(p0, np.random.default_rng(8), 0.2)
    fit = diff.Fit(rs)
    fit.targets(truth)
    targets = [np.nan_to_num(r.ForwardLinear(truth)) for r in rs]
    lr = 1e-2
    p1, _ = fit.run(p0, steps=1, lr=lr, groups=groups)
    p2, hist = fit.run(p0, steps=2, lr=lr, groups=groups)
    l0, G0 = _summed_backward(rs, p0, targets)
    l1, G1 = _summed_backward(rs, p1, targets)
    assert abs(hist[0] - l0) <= 1e-4 * l0 and abs(hist[1] - l1) <= 1e-4 * l0, (hist, l0, l1)
    for n in diff.DiffParams.NAMES:
        if n == "normal":
            continue
        if n not in groups:
            assert np.array_equal(getattr(p2, n), getattr(p0, n)), n
            continue
        base = getattr(p0, n).astype(np.float64).reshape(-1)
        th, m, v = np.zeros_like(base), np.zeros_like(base), np.zeros_like(base)
        g0 = getattr(G0, n).astype(np.float64).reshape(-1) * base
        g1 = getattr(G1, n).astype(np.float64).reshape(-1) * base
        th, m, v = _adam64(th, m, v, g0, 1, lr)
        th, m, v = _adam64(th, m, v, g1, 2, lr)
        got = getattr(p2, n).astype(np.float64).reshape(-1)
        big = (np.abs(g0) > 1e-2 * np.abs(g0).max()) & (np.abs(g1) > 1e-2 * np.abs(g1).max())
        assert big.any(), n
        # (the bar of test_two_steps_follow_host_adam)
        assert np.abs(got - base * (1 + th))[big].max() <= 1e-3 * lr * np.abs(base[big]).max() + 1e-6, n
        # a parameter no pixel sees stays put
        unseen = (g0 == 0) & (g1 == 0)
        assert np.array_equal(got[unseen], base[unseen]), n
    fit.free()
    gs.free()
