"""Small jobs packed sixty-four to a wave in the raster, on the MI355X against
the oracle bit for bit: with nothing drawn by the setup, one raster workgroup a
CU (64 waves a queue) and job counts below, around and above the eight a wave
from which it packs them; small and large jobs in one wave; the view, the shadow
maps and the exact-order pass after a NaN depth."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import cases

pytestmark = pytest.mark.gpu


def _same(r, fr):
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    assert np.array_equal(order, fr.vis_order)
    a, b = r.read(abi.PRH_BUF_DEPTH), fr.depth.reshape(r.H, r.W)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])
    assert np.array_equal(r.image(), fr.image)


# some 400 of a sphere's triangles face a view: 8192 jobs, 8 a wave, lie between
# 18 and 30 of them in the view, and five maps together get five times as many
@pytest.mark.parametrize("spheres", [2, 5, 18, 24, 30, 90])
@pytest.mark.parametrize("direct", [0, 3])
def test_view_and_maps(device, orc, spheres, direct):
    s = scenes.c2_scale(seed=7, width=320, height=240, n_spheres=spheres, grid=12, shadow_size=200, ao=False)
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    for tile in (16, 8):
        r.set_tuning(main_direct_max=direct, shadow_direct_max=direct, raster_wg_per_cu=1, raster_tile=tile)
        r.render_device()
        _same(r, fr)
        got = r.read(abi.PRH_BUF_SHADOW).reshape(-1)
        assert np.array_equal(got.view(np.uint32), fr.shadow_maps[: got.size].view(np.uint32))
    render.render_batch([r])
    _same(r, fr)
    r.free()


@pytest.mark.parametrize("n", [7000, 9000, 20000])
def test_exact_order(device, orc, n):
    side = 160
    Y = -0.34375  # 80 Y + 80 = 52.5, a row of pixel centres: 0/0 there
    rng = np.random.default_rng(n)
    c = np.concatenate([rng.uniform(-0.9, 0.9, (n, 2)), 0.3 * rng.uniform(-1, 1, (n, 1)), np.ones((n, 1))], 1)
    d = np.zeros((n, 3, 4))
    d[:, 1, 0] = d[:, 2, 1] = 0.03 * np.exp(rng.uniform(np.log(0.3), np.log(4), n))  # 1 to 10 pixels a side
    P = np.concatenate([[[[-0.5, Y, 0.5, 1], [0.5, Y, 0.5, 1], [0.0, Y, -0.5, 1]]], c[:, None, :] + d])
    P[..., :2] = np.clip(P[..., :2], -0.99, 0.99)
    s = cases._scene(P.reshape(-1, 4), np.arange(3 * (n + 1), dtype=np.int32).reshape(-1, 3), [0] + [-1] * n, side, side,
                     cases.ORTHO)
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    r.set_tuning(raster_wg_per_cu=1)
    r.render_device()
    assert r.stats().nan_rerun == 1
    _same(r, fr)
    r.free()
