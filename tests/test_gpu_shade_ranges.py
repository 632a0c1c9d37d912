"""k_shade's roots and quotients without scaling, and the waves that leave
them (an operand outside their range in some lane), on the MI355X against the
oracle, bit for bit: lights far off, next to and in the surface, intensities
of 0, tiny, huge, infinite and NaN, worlds 2^-45 and 2^45 the size, flat
shading, vertex colours beside materials."""
import numpy as np
import pytest

from polyred_amd import abi, render, scenes

from . import cases

pytestmark = pytest.mark.gpu


def _same(device, orc, s):
    fr = orc.render(s)
    r = render.renderer_for(s, device, keep_linear=True)
    r.render_device()
    assert np.array_equal(r.read(abi.PRH_BUF_PREGAMMA).reshape(-1, 4), fr.pregamma.reshape(-1, 4))
    a, b = r.read(abi.PRH_BUF_LINEAR).reshape(-1), fr.linear.reshape(-1)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)], b[~np.isnan(b)])
    assert np.array_equal(r.image(), fr.image)
    r.free()


def _lights(kind):
    L = scenes.Light
    near = dict(position=(0.0, 0.0, 0.2))  # in the large triangle's plane
    return {
        "plain": [L(position=(1.0, 2.0, 3.0)), L(position=(-2.0, 0.5, 1.0), intensity=0.0)],
        "near": [L(**near), L(position=(0.0, 0.0, 0.2 + 1e-12)), L(position=(0.1, 0.1, 0.25))],
        "far": [L(position=(3e9, -2e9, 5e9), intensity=1e10), L(position=(1e25, 1e25, 1e25), intensity=1e25)],
        "tiny": [L(position=(1.0, 2.0, 3.0), intensity=1e-30), L(position=(0.0, 2.0, 2.0), intensity=2.0)],
        "huge": [L(position=(1.0, 2.0, 3.0), intensity=1e30), L(position=(0.0, 2.0, 2.0), intensity=3e38)],
        "wild": [L(position=(1.0, 2.0, 3.0), intensity=float("inf")), L(position=(float("nan"), 0.0, 1.0)),
                 L(position=(0.0, 2.0, 2.0), intensity=float("nan"))],
    }[kind]


@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("kind", ["plain", "near", "far", "tiny", "huge", "wild"])
def test_lights(device, orc, kind, flat):
    s = cases.big_triangle(70, 41)
    s.lights = _lights(kind)
    for m in s.materials:
        m.flat_shading = flat
    _same(device, orc, s)


@pytest.mark.parametrize("scale", [2.0 ** -45, 2.0 ** -20, 2.0 ** 20, 2.0 ** 45])
def test_world_sizes(device, orc, scale):
    s = cases.big_triangle(70, 41)
    for m in s.meshes:
        m.pos[:, :3] *= np.float32(scale)
    c = s.camera
    for k in ("near", "far"):
        c[k] *= scale
    c["position"] = tuple(scale * v for v in c["position"])
    s.lights = [scenes.Light(position=(1.0 * scale, 2.0 * scale, 3.0 * scale), intensity=scale)]
    _same(device, orc, s)
