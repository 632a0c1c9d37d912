"""The antialiased frame's resize on the MI355X against the oracle, byte for
byte: tiles of 64 positions by 32 rows (from 2^17 outputs and up to 8 taps)
around their sides, and a thread a pixel below that and for longer filters, in
a frame of its own and in a recorded batch that holds both."""
import numpy as np
import pytest

from polyred_amd import render, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,m", [(1, 1, 2), (33, 65, 3), (64, 32, 5), (512, 128, 2), (513, 257, 2), (700, 97, 3),
                                   (65, 1021, 2), (300, 129, 4), (260, 130, 5)])
def test_resize(device, orc, w, h, m):
    s = scenes.textured(seed=4, width=w, height=h)
    s.msaa = m
    fr = orc.render(s)
    r = render.renderer_for(s, device)
    r.render_device()
    assert np.array_equal(r.image(), fr.image)
    t = scenes.textured(seed=5, width=40, height=30)
    t.msaa = 2
    q = render.renderer_for(t, device)
    render.render_batch([q, r])
    assert np.array_equal(r.image(), fr.image) and np.array_equal(q.image(), orc.render(t).image)
    q.free()
    r.free()
