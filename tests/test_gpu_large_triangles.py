"""The adjoint's vertex gradients where a triangle covers many pixels: waves of
one triangle, of a few and of many (a triangle with eight lanes of a wave is
summed over it), tables that hold few vertices to the end and ones that fill
and are emptied between, on the MI355X through the C ABI against the FP64
reference at test_gpu_adjoint_sizes' bars; and what large triangles cost."""
import numpy as np
import pytest

import oracle
from polyred_amd import abi, diff, render, scenes

pytestmark = pytest.mark.gpu


def _plane(n, w, h):
    s = scenes.c4_adjoint(width=w, height=h, n_spheres=1)
    g = scenes.grid_plane(n, 14.0, -2.0)
    g.col = np.random.default_rng(n).integers(60, 255, g.col.shape).astype(np.uint8)
    s.meshes, s.obj_mesh = [g], np.array([0])
    s.obj_model = np.eye(4, dtype=np.float32).reshape(1, 16)
    s.obj_mat_base = np.array([0])
    s.camera = dict(position=(0.0, 16.0, 1.0), target=(0.0, -2.0, 0.0), fov=60.0, near=0.1, far=100.0)
    return s


@pytest.mark.parametrize("w,h", [(64, 64), (300, 201)])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 16, 41, 100])
@pytest.mark.parametrize("normals", [False, True])
def test_gradients(device, orc, w, h, n, normals):
    s = _plane(n, w, h)
    r = render.renderer_for(s, device)
    r.render_device()
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    p = diff.scene_params(s)
    if normals:
        N = np.random.default_rng(7).normal(0, 0.2, (len(p.albedo), 3)) + [0, 1, 0]
        p.normal = N.astype(np.float32)
    target = np.nan_to_num(0.5 * r.ForwardLinear(p)).astype(np.float32)
    loss, g = r.Backward(p, target)
    ref_loss, ref, gref = oracle.diff(s, order, p, target.astype(np.float64))
    assert (~np.isnan(ref)).all(-1).sum() > w * h // 2
    assert abs(loss - ref_loss) <= 1e-4 * ref_loss
    for name in diff.DiffParams.NAMES:
        a = np.asarray(getattr(g, name), np.float64).reshape(-1)
        b = np.asarray(gref[name], np.float64).reshape(-1)
        assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(b) + 1e-12, name
    r.free()


def test_two_triangles_cost_no_more_than_twice_two_thousand(device):
    """Without the sum over the wave and the table's later flush: 3.3 times."""
    ms = {}
    for n in (1, 32):
        s = _plane(n, 1024, 1024)
        r = render.renderer_for(s, device)
        r.render_device()
        p = diff.scene_params(s)
        target = np.zeros((1024, 1024, 3), np.float32)
        best = np.inf
        for _ in range(8):
            r.Backward(p, target)
            best = min(best, r.stats().ms_diff)
        ms[n] = best
        r.free()
    print("ms", ms)
    assert ms[1] <= 2.0 * ms[32], ms
