"""The differentiable shading's geometry is the forward pass's, in its own
float32: barycentrics at the pixel centre (areas as float64 FMAs of a rounded
product), perspective weights.  Needles -- triangles as long as the view and a
fraction of a pixel wide -- have areas far below the products they are the
differences of, so a barycentric of any other rounding is another number
there.  On the MI355X through the C ABI against the FP64 reference, whose
geometry is the forward's.

Without lights the linear colour is ambient * sum w_k A_k with positive
albedo, six roundings of at most 2^-24 each (three products or FMAs, the
ambient's float32 sum, its product, the result), so 2^-21 relative is above
any float32 evaluation of it."""
import numpy as np
import pytest

import oracle
from polyred_amd import abi, diff, render

from . import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("persp", [True, False])
@pytest.mark.parametrize("seed", range(4))
def test_needles(device, orc, seed, persp):
    rng = np.random.default_rng(seed)
    n, side = 400, 256
    a = rng.uniform(-0.9, 0.9, (n, 2))
    b = rng.uniform(-0.9, 0.9, (n, 2))
    d = b - a
    perp = np.stack([-d[:, 1], d[:, 0]], 1) / np.linalg.norm(d, axis=1, keepdims=True)
    width = 2 / side * np.exp(rng.uniform(np.log(0.01), np.log(2.0), (n, 1)))  # 1/100 to 2 pixels
    P = np.ones((n, 3, 4))
    for k, q in enumerate((a, b, a + width * perp)):
        P[:, k, :2] = q
    P[:, :, 2] = rng.uniform(-0.5, 0.5, (n, 1)) + (0.2 * rng.uniform(-1, 1, (n, 3)) if persp else 0)
    tri = np.arange(3 * n).reshape(-1, 3)
    # facing the camera at z = 3
    col = np.concatenate([rng.integers(40, 256, (3 * n, 3)), np.full((3 * n, 1), 255)], 1).astype(np.uint8)
    cam = dict(position=(0.0, 0.0, 3.0), fov=40.0, near=0.1, far=100.0) if persp else cases.ORTHO
    s = cases._scene(P.reshape(-1, 4), tri, [0] * n, side, side, cam, lights=[], col=col)
    r = render.renderer_for(s, device)
    r.render_device()
    vis = r.read(abi.PRH_BUF_VIS)
    order = (vis & np.uint64(0xFFFFFFFF)).astype(np.uint32)
    order[vis == np.uint64(0xFFFFFFFFFFFFFFFF)] = 0xFFFFFFFF
    p = diff.scene_params(s)
    lin = r.ForwardLinear(p)
    _, ref, _ = oracle.diff(s, order, p)
    ok = ~np.isnan(ref)
    assert ok.sum() > 3000 and np.array_equal(ok, ~np.isnan(lin))
    err = np.abs(lin[ok].astype(np.float64) - ref[ok]) / ref[ok]
    assert err.max() <= 2.0 ** -21, err.max()
    r.free()
