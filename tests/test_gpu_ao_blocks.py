"""k_ao's marches by blocks of eight taps on the MI355X against the oracle, bit
for bit: frames around the blocks' and the bounds' sides (rows and columns in
fours, chunks of 64 pixels, 256-column workgroups), narrower or lower than a
march, the rows and columns where the axis directions' taps change line, a
frame past the tables' 4096, in one stream, two, and a recorded batch."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import golden_cases

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 2), (64, 1), (1, 70), (7, 9), (65, 13), (103, 104), (130, 97), (257, 12), (300, 259), (523, 31)]


def _scene(w, h, kind):
    if kind == "plane":
        s = golden_cases.c1_shadow_ao()
        s.width, s.height = w, h
        return s
    return scenes.c2_scale(seed=w + h, width=w, height=h, n_spheres=40, grid=8, shadow_size=64)


def _same(r, fr):
    assert np.array_equal(r.read(abi.PRH_BUF_PREGAMMA).reshape(-1, 4), fr.pregamma.reshape(-1, 4))
    assert np.array_equal(r.image(), fr.image)


@pytest.mark.parametrize("kind", ["plane", "spheres"])
@pytest.mark.parametrize("w,h", SIZES)
def test_frame(device, orc, w, h, kind):
    s = _scene(w, h, kind)
    fr = orc.render(s)
    r = render.renderer_for(s, device, keep_linear=True)
    for overlap in (0, 1):
        r.set_tuning(overlap_shadows=overlap)
        r.render_device()
        _same(r, fr)
    r.free()


def test_past_the_tables(device, orc):
    s = _scene(4099, 5, "plane")
    r = render.renderer_for(s, device, keep_linear=True)
    r.render_device()
    _same(r, orc.render(s))
    r.free()


def test_batch(device, orc):
    """Views with and without the tables (and so the bounds' kernel) in one."""
    ss = [_scene(w, h, k) for w, h, k in ((130, 97, "spheres"), (4099, 5, "plane"), (65, 13, "plane"))]
    rs = [render.renderer_for(s, device, keep_linear=True) for s in ss]
    for order in (rs, rs[::-1]):
        render.render_batch(order)
        for s, r in zip(ss, rs):
            _same(r, orc.render(s))
    for r in rs:
        r.free()
