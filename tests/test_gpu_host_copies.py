"""Copies to and from the caller's memory through the library's page-locked
stage on the MI355X: sizes around its chunks and past the stage, unaligned
addresses, ordinary and page-locked memory alike, and contexts in two threads."""
import ctypes as C
import threading

import numpy as np
import pytest

from polyred_amd import abi, diff, render, scenes

pytestmark = pytest.mark.gpu

STAGE = 8 << 20
CHUNK = STAGE // 32


@pytest.mark.parametrize("w,h", [(1, 1), (3, 1), (256, 255), (256, 256), (257, 256), (1024, 192), (2048, 1024),
                                 (2049, 1025)])
def test_image_in_ordinary_memory(device, w, h):
    """(256x256 RGBA8 is a chunk, 2048x1024 the stage)"""
    s = scenes.c1_plain(width=w, height=h)
    r = render.renderer_for(s, device)
    r.render_device()
    want = r.image(render.pinned_array((h, w, 4)))
    raw = np.zeros(4 * w * h + 64, np.uint8)
    for shift in (0, 1, 4, 8, 15):
        raw[:] = 0xA5
        out = raw[shift:shift + 4 * w * h]
        abi.check(r._lib.prh_read_image(r.handle, out.ctypes.data, out.nbytes), "prh_read_image")
        assert np.array_equal(out.reshape(h, w, 4), want)
        assert (raw[:shift] == 0xA5).all() and (raw[shift + 4 * w * h:] == 0xA5).all()
    vis = r.read(abi.PRH_BUF_VIS)  # twice the bytes
    pin = render.pinned_array((8 * w * h,))
    abi.check(r._lib.prh_read_buffer(r.handle, abi.PRH_BUF_VIS, pin.ctypes.data, pin.nbytes), "prh_read_buffer")
    assert np.array_equal(vis.reshape(-1), pin.view(np.uint64))
    r.free()


def test_target_past_the_stage(device):
    """A target (and a forward result) of more bytes than the stage holds."""
    s = scenes.c4_adjoint(seed=2, width=1003, height=901, n_spheres=6)
    r = render.renderer_for(s, device)
    r.render_device()
    p = diff.scene_params(s)
    lin = r.ForwardLinear(p)
    assert lin.nbytes > STAGE
    assert np.array_equal(np.nan_to_num(lin), np.nan_to_num(r.ForwardLinear(p)))
    loss, g = r.Backward(p, np.nan_to_num(lin))  # the target every pixel has
    assert loss == 0.0 and all(not np.any(a) for a in g.arrays().values())
    r.free()


def test_contexts_in_two_threads():
    def work(seed, out):
        d = render.Device(0)
        s = scenes.c4_adjoint(seed=seed, width=200, height=150, n_spheres=6)
        r = render.renderer_for(s, d)
        p = diff.scene_params(s)
        for _ in range(20):
            r.render_device()
            out.append((r.image().copy(), np.nan_to_num(r.ForwardLinear(p))))
        r.free()

    res = [[], []]
    ts = [threading.Thread(target=work, args=(k, res[k])) for k in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    for out in res:
        assert len(out) == 20
        for im, lin in out[1:]:
            assert np.array_equal(im, out[0][0]) and np.array_equal(lin, out[0][1])
