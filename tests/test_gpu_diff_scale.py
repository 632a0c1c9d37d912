"""The division of the differentiable shading's sums by 255 leaves no bias: a
quotient of a material's colour rounded before the pixel's sums would be the
same for all of its pixels, and the sums over pixels (the loss, the material
gradients) would keep it.  On the MI355X through the C ABI against the FP64
reference, with colours whose float32 quotient by 255 is over 5e-8 off in one
direction.

Bars: the mean relative error of n pixels whose roundings are their own, some
20 of at most 2^-24 each (under 2^-25 rms), is below 2^-25 sqrt(20 / n); n is
taken as a twentieth of the pixels, as neighbours share vertices: some 4e-9
for the 20 thousand pixels and more here, a twelfth of the quotient's error."""
import numpy as np
import pytest

import oracle
from polyred_amd import abi, diff, render, scenes

pytestmark = pytest.mark.gpu


def _off(x):
    """The relative error of float32(x / 255)."""
    q = np.float32(np.float64(np.float32(x)) / 255)
    return float((np.float64(q) - np.float64(np.float32(x)) / 255) / (np.float64(np.float32(x)) / 255))


@pytest.mark.parametrize("what", ["kd", "ks"])
@pytest.mark.parametrize("sign", [1, -1])
def test_no_bias(device, orc, what, sign):
    value = next(v for v in np.arange(128, 150, 1 / 64) if sign * _off(v) > 5e-8)
    s = scenes.c4_adjoint(seed=5, width=512, height=512, n_spheres=104)
    r = render.renderer_for(s, device)
    r.render_device()
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    s.ambient = [0.0]
    r.free()
    r = render.renderer_for(s, device)
    r.render_device()
    p = diff.scene_params(s)
    p.kd[:] = value if what == "kd" else 0.0
    p.ks[:] = value if what == "ks" else 0.0
    p.shininess[:] = 4.0
    lin = r.ForwardLinear(p).astype(np.float64)
    _, ref, _ = oracle.diff(s, order, p)
    ok = ref > 1.0
    n = int(ok.all(-1).sum())
    assert n > 20_000
    bias = float(((lin - ref)[ok] / ref[ok]).mean())
    assert abs(bias) <= 2.0 ** -25 * np.sqrt(20 / (n / 20)), (bias, _off(value))
    # the loss and the gradient against a target of half the colour
    target = np.nan_to_num(0.5 * ref).astype(np.float32)
    loss, g = r.Backward(p, target)
    ref_loss, _, gref = oracle.diff(s, order, p, target.astype(np.float64))
    bar = 3 * 2.0 ** -25 * np.sqrt(20 / (n / 20))  # (a square and its product with the residual; bright pixels count more)
    assert abs(loss - ref_loss) <= 2 * bar * ref_loss, (loss / ref_loss - 1, _off(value))
    r.free()
