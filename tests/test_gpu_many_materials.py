"""The adjoint past 585 materials, whose sums are kept in bins found by open
addressing (512 a workgroup, eight probes) on the MI355X through the C ABI:
materials spread over the bins, all meeting at one bin so that some find none,
and more of them than bins, against the FP64 reference at test_gpu_adjoint_sizes'
bars; and what a step costs there."""
import time

import numpy as np
import pytest

from polyred_amd import diff, render, scenes

from .test_gpu_adjoint_sizes import _check, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_mats,of", [(586, lambda i: i * 13 % 586), (8000, lambda i: 512 * (i % 15)),
                                       (8000, lambda i: 512 * (i % 15) + i % 3), (3000, lambda i: i * 997 % 3000)])
def test_gradients(device, orc, n_mats, of):
    s = _scene(90, 70, n_mats=n_mats)
    s.obj_mat_base = np.array([of(i) for i in range(len(s.obj_mat_base))])
    assert _check(device, s) > 1000


def test_more_than_bins(device, orc):
    """A material per triangle: thousands in the view."""
    s = _scene(200, 160, n_mats=9600)
    mesh = s.meshes[0]
    mesh.mat = np.arange(len(mesh.tri), dtype=np.int32)
    s.obj_mat_base = (np.arange(len(s.obj_mat_base)) % 10) * len(mesh.tri)
    assert 10 * len(mesh.tri) <= 9600
    assert _check(device, s) > 1000


def test_a_step_costs_no_tenfold(device):
    times = []
    for n_mats in (8, 700):
        s, views = scenes.c5_inverse(seed=5, n_views=4, n_spheres=60, min_side=200, max_side=400, shadow_size=256)
        proto = s.materials
        s.materials = [proto[i % len(proto)] for i in range(n_mats)]
        s.obj_mat_base = np.arange(len(s.obj_mat_base)) * 37 % n_mats
        gs, rs = render.views_of(s, views, device)
        for r in rs:
            r.render_device()
        p = diff.scene_params(s)
        fit = diff.Fit(rs)
        fit.targets(p)
        start = diff.perturb(p, np.random.default_rng(1), 0.1)
        best = np.inf
        for _ in range(5):
            t0 = time.perf_counter()
            fit.run(start, steps=10)
            best = min(best, time.perf_counter() - t0)
        times.append(best)
        fit.free()
        gs.free()
    assert times[1] <= 10 * times[0], times
