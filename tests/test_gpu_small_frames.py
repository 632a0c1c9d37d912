"""Frames without AO on the MI355X against the oracle, bit for bit, around the
size up to which the uncovered pixels shade pixel (0,0) themselves (2^17
pixels): pixel (0,0) covered and not, with and without materials, one stream
and two, and in a recorded batch; and their depth, which the shading writes."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import cases, golden_cases

pytestmark = pytest.mark.gpu


def _scene(kind, w, h):
    if kind == "textured":  # pixel (0,0) covered from the larger frames on
        return scenes.textured(seed=3, width=w, height=h)
    if kind == "bare":  # without materials
        s = cases.no_materials()
    elif kind == "layers":  # pixel (0,0) uncovered, except in a frame of one pixel
        return cases.stacked_layers(n_layers=3, width=w, height=h)
    else:  # shadows, pixel (0,0) as in the textured scene
        s = golden_cases.c1_shadow_ao()
        for m in s.materials:
            m.ambient_occlusion = False
    s.width, s.height = w, h
    return s


def _same(r, fr):
    a = r.read(abi.PRH_BUF_DEPTH).reshape(-1)
    assert np.array_equal(a.view(np.uint32), fr.depth.reshape(-1).view(np.uint32))
    assert np.array_equal(r.read(abi.PRH_BUF_PREGAMMA).reshape(-1, 4), fr.pregamma.reshape(-1, 4))
    la, lb = r.read(abi.PRH_BUF_LINEAR).reshape(-1), fr.linear.reshape(-1)
    assert np.array_equal(np.isnan(la), np.isnan(lb)) and np.array_equal(la[~np.isnan(la)], lb[~np.isnan(lb)])
    assert np.array_equal(r.image(), fr.image)


@pytest.mark.parametrize("kind", ["bare", "textured", "layers", "plane"])
@pytest.mark.parametrize("w,h", [(1, 1), (17, 5), (512, 256), (513, 256)])
def test_frame(device, orc, kind, w, h):
    s = _scene(kind, w, h)
    fr = orc.render(s)
    r = render.renderer_for(s, device, keep_linear=True)
    for overlap in (0, 1):
        r.set_tuning(overlap_shadows=overlap)
        r.render_device()
        _same(r, fr)
    q = render.renderer_for(_scene("plane", 40, 30), device, keep_linear=True)
    render.render_batch([q, r])
    _same(r, fr)
    q.free()
    r.free()
