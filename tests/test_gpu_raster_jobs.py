"""The raster's jobs (rectangles of a large primitive's pixel box, two raster
tiles a side) on the MI355X against the oracle, bit for bit: images around the
jobs' sides, every tile side, nothing, some and everything drawn by the setup;
queues that overflow in the plain pass, in the shadow passes, and only in the
exact-order pass after a NaN depth."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import cases

pytestmark = pytest.mark.gpu


def _order(r):
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    return order


def _same(r, fr):
    assert np.array_equal(_order(r), fr.vis_order)
    a, b = r.read(abi.PRH_BUF_DEPTH), fr.depth.reshape(r.H, r.W)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])
    assert np.array_equal(r.image(), fr.image)


@pytest.mark.parametrize("w,h", [(1, 1), (15, 17), (16, 16), (31, 33), (64, 64), (65, 129), (130, 31), (193, 97)])
@pytest.mark.parametrize("tile", [8, 16, 32])
def test_job_edges(device, orc, w, h, tile):
    s = cases.stacked_layers(n_layers=3, width=w, height=h)
    s.shadow_size = w + 7  # maps of another size
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    for small in (0, 48, 256):
        r.set_tuning(raster_tile=tile, main_direct_max=small, shadow_direct_max=small)
        r.render_device()
        _same(r, fr)
        assert np.array_equal(r.read(abi.PRH_BUF_SHADOW)[0].reshape(-1), fr.shadow_maps.reshape(-1))
    s = cases.big_triangle(w, h)  # clipped pieces
    fr = orc.render(s)
    q = render.renderer_for(s, device)
    for small in (0, 48):
        q.set_tuning(raster_tile=tile, main_direct_max=small)
        q.render_device()
        _same(q, fr)
    r.free()
    q.free()


def test_statistics_count_primitives_and_tiles(device):
    """n_prims and n_bin_pairs from their definition: screen-facing quads in
    an orthographic view whose corners are known pixels."""
    side, n = 96, 5
    P, tri = [], []
    for k in range(n):
        x0, x1 = -1 + 2 * (8 * k + 0.25) / side, -1 + 2 * (8 * k + 40.25) / side
        b = len(P)
        P += [[x0, x0, 0, 1], [x1, x0, 0, 1], [x1, x1, 0, 1]]
        tri += [[b, b + 1, b + 2]]
    s = cases._scene(P, tri, [0] * n, side, side, cases.ORTHO)
    r = render.renderer_for(s, device)
    r.set_tuning(main_direct_max=0)
    r.render_device()
    st = r.stats()
    # the box narrowed to the pixel centres in [min - 0.24, max + 0.24]
    want = 0
    for k in range(n):
        a, b = 8 * k + 0.25, 8 * k + 40.25
        lo, hi = int(np.ceil(a - 0.74)), int(np.floor(b - 0.26))
        want += ((hi >> 4) - (lo >> 4) + 1) ** 2
    assert (st.n_prims, st.n_bin_pairs, st.n_clipped) == (n, want, 0)
    r.set_tuning(main_direct_max=256)  # boxes of 41 x 41: none drawn by the setup
    r.render_device()
    assert (r.stats().n_prims, r.stats().n_bin_pairs) == (n, want)
    r.free()


def test_exact_order_pass_outgrows_the_queues(device, orc):
    """Ten triangles that cover the screen make 1000 jobs of 16 x 16, which
    fit; the 300 small ones beside them are drawn by the setup in the plain
    pass and are jobs in the exact-order pass, which the first capacity
    (triangles / 16 + pixels / 256 + 1024 a queue) does not hold."""
    side = 160
    Y = -0.34375  # 80 Y + 80 = 52.5, a row of pixel centres: 0/0 there
    P, tri = [[-0.5, Y, 0.5, 1], [0.5, Y, 0.5, 1], [0.0, Y, -0.5, 1]], [[0, 1, 2]]
    for k in range(10):
        b = len(P)
        P += [[-0.99, -0.99, -0.01 * k, 1], [0.99, -0.99, -0.01 * k, 1], [0.0, 0.99, -0.01 * k, 1]]
        tri += [[b, b + 1, b + 2]]
    rng = np.random.default_rng(3)
    for k in range(240):
        x, y, z = rng.uniform(-0.9, 0.9, 3)
        b = len(P)
        P += [[x, y, 0.3 * z, 1], [x + 0.03, y, 0.3 * z, 1], [x, y + 0.03, 0.3 * z, 1]]
        tri += [[b, b + 1, b + 2]]
    s = cases._scene(P, np.asarray(tri, np.int32), [0] * 11 + [-1] * 240, side, side, cases.ORTHO)
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    r.set_tuning(raster_tile=8)
    for _ in range(2):
        r.render_device()
        assert r.stats().nan_rerun == 1
        _same(r, fr)
    render.render_batch([r])
    _same(r, fr)
    r.free()


@pytest.mark.parametrize("far", [1e4, 3e8, 3e9, 1e12, 1e30])
def test_boxes_past_32_bits(device, orc, far):
    """Triangles whose screen coordinates in the view and in the shadow maps
    lie within and beyond what 32-bit pixel boxes hold."""
    s = cases.shadow_footprint()
    for m in s.meshes:
        p = m.pos[:, :2]
        p[np.abs(p) >= np.abs(p).max() * 0.99] *= np.float32(far)  # the ground's corners
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    try:
        r.render_device()
    except abi.PrhError as e:  # (areas that overflow: a NaN depth in a shadow pass is refused)
        assert e.code == abi.PRH_E_UNSUPPORTED and far in (3e9, 1e12)
        r.free()
        return
    _same(r, fr)
    got = r.read(abi.PRH_BUF_SHADOW).reshape(-1)
    assert np.array_equal(got.view(np.uint32), fr.shadow_maps[: got.size].view(np.uint32))
    r.free()


@pytest.mark.parametrize("knob", [0, 15, 16, 47, 48, 49, 256])
def test_threshold_by_frame_size(device, orc, knob):
    """The setup's threshold in a small frame (16 with the knob at its default,
    else the knob's) and in a batch: the same frame, and the same statistics,
    which go by the knob."""
    s = scenes.c2_scale(seed=3, width=200, height=150, n_spheres=20, grid=6, shadow_size=64, ao=False)
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    r.set_tuning(main_direct_max=knob)
    r.render_device()
    _same(r, fr)
    a = r.stats()
    render.render_batch([r])
    _same(r, fr)
    b = r.stats()
    assert (a.n_prims, a.n_bin_pairs, a.n_clipped) == (b.n_prims, b.n_bin_pairs, b.n_clipped)
    r.free()
