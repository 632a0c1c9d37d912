"""A frame whose raster jobs no memory holds (450 thousand triangles across the
view in 16x16 rectangles: 350 GB of them) is refused, and so is the next one:
the renderer is left with the buffers' old capacities and allocates those
again before it launches anything.  With 64x64 rectangles (a sixteenth of the
jobs) the same renderer then draws the frame: the triangles are one triangle
repeated, of which the first wins everywhere.  The other renderers of the
context, alone and in a batch with it, are not touched."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import cases

pytestmark = pytest.mark.gpu

SIDE = 2048


def _needle(n):
    """One needle from corner to corner, n times: it covers few pixels, its
    pixel box all of them."""
    P = [[-0.99, -0.99, 0, 1], [0.99, 0.985, 0, 1], [0.985, 0.99, 0, 1]]
    return cases._scene(P, np.tile(np.array([[0, 1, 2]], np.int32), (n, 1)), np.zeros(n, np.int32), SIDE, SIDE,
                        cases.ORTHO)


def test_growth_past_the_memory(device, orc):
    small = scenes.tiny(3, width=64, height=48, n_tris=10)
    want = orc.render(small)
    q = render.renderer_for(small, device)
    one = render.renderer_for(_needle(1), device)
    one.render_device()
    vis = one.read(abi.PRH_BUF_VIS)
    assert (vis != np.uint64(0xFFFFFFFFFFFFFFFF)).sum() > 500
    r = render.renderer_for(_needle(450_000), device)
    r.set_tuning(raster_tile=8, main_direct_max=0)
    for draw in (r.render_device, r.render_device, lambda: render.render_batch([q, r]),
                 lambda: render.render_batch([q, r], graph=True), lambda: render.render_batch([q, r], streams=True)):
        with pytest.raises(abi.PrhError) as e:
            draw()
        assert e.value.code == abi.PRH_E_NOMEM
        assert np.array_equal(q.Render(), want.image)
    r.set_tuning(raster_tile=32)
    r.render_device()
    assert np.array_equal(r.read(abi.PRH_BUF_VIS), vis)
    for x in (r, one, q):
        x.free()


def test_counts_past_31_bits(device):
    """2.3 million triangles of 16384 jobs: 2.36e9 a queue, past what 32-bit
    counts tell from a place in the queue."""
    r = render.renderer_for(_needle(2_300_000), device)
    r.set_tuning(raster_tile=8, main_direct_max=0)
    for draw in (r.render_device, lambda: render.render_batch([r])):
        with pytest.raises(abi.PrhError) as e:
            draw()
        assert e.value.code == abi.PRH_E_NOMEM
    r.free()
