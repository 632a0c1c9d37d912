"""Screen coordinates within and beyond what 32-bit pixel boxes hold, each with
one expected outcome, on the MI355X: without shadow maps every frame equals the
oracle's; with them too, but for coordinates of 3e9 and 1e12, where areas
overflow to a NaN depth in a shadow pass, which is refused."""
import numpy as np
import pytest

from polyred_amd import abi, render

from . import cases

pytestmark = pytest.mark.gpu


def _scene(far, shadows):
    s = cases.shadow_footprint()
    for m in s.meshes:
        p = m.pos[:, :2]
        p[np.abs(p) >= np.abs(p).max() * 0.99] *= np.float32(far)  # the ground's corners
    s.shadow_map = shadows
    for light in s.lights:
        light.cast_shadow = light.cast_shadow and shadows
    return s


def _same(r, fr):
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    assert np.array_equal(order, fr.vis_order)
    assert np.array_equal(r.read(abi.PRH_BUF_DEPTH).view(np.uint32), fr.depth.reshape(r.H, r.W).view(np.uint32))
    assert np.array_equal(r.image(), fr.image)


@pytest.mark.parametrize("far", [1e4, 3e8, 1e9, 3e9, 1e12, 1e30])
def test_view(device, orc, far):
    s = _scene(far, False)
    r = render.renderer_for(s, device)
    r.render_device()
    _same(r, orc.render(s))
    r.free()


@pytest.mark.parametrize("far,refused", [(1e4, False), (3e8, False), (3e9, True), (1e12, True), (1e30, False)])
def test_shadow_maps(device, orc, far, refused):
    s = _scene(far, True)
    r = render.renderer_for(s, device)
    if refused:
        with pytest.raises(abi.PrhError) as e:
            r.render_device()
        assert e.value.code == abi.PRH_E_UNSUPPORTED
    else:
        fr = orc.render(s)
        r.render_device()
        _same(r, fr)
        got = r.read(abi.PRH_BUF_SHADOW).reshape(-1)
        assert np.array_equal(got.view(np.uint32), fr.shadow_maps[: got.size].view(np.uint32))
    r.free()
