"""Performance cases: the calls a program that uses polyred_amd makes, over
the sizes and options it makes them with.

  frame    one (*Renderer).Render(): shadow passes, forward raster, deferred
           shading, gamma, and the image on the host
  batch    one frame of many independent views in one submission, every image
           read back
  adjoint  one step of an inverse-rendering program that moves the geometry:
           a frame, then the loss and every gradient at its visibility
  relight  the linear shading of a frame already drawn, at new parameters
  fit      a burst of Adam steps over many views at fixed visibility

The scenes are this package's generators (polyred_amd/scenes.py), seeded.
exact() restates the differentiable shading in float64 torch.
"""
import math

import numpy as np
import torch

from polyred_amd import diff, render, scenes

_dev = None


def _device():
    """The program's one opened GPU."""
    global _dev
    if _dev is None:
        _dev = render.Device(0)
    return _dev


# ------------------------------------------------------------------- cases
def listed():
    scale = dict(kind="frame", scene="scale", msaa=1, ao=True, shadows=True, grid=200, spheres=1000, shadow_size=2048,
                 pinned=True)
    return [
        # a thumbnail or a test image: one object on a ground plane; launches
        # and the call itself are all there is
        dict(name="plain_256", kind="frame", scene="plain", width=256, height=256, msaa=1, ao=False, shadows=False,
             pinned=False),
        # a small asset at polyred's default size (800x600), mip-mapped
        # textures, two shadow-casting lights with framebuffer-sized maps,
        # 2x antialiasing
        dict(name="textured_800x600_msaa2", kind="frame", scene="textured", width=800, height=600, msaa=2, ao=False,
             shadows=True, pinned=False),
        # a preview of a large scene
        dict(scale, name="scale_480x270", width=480, height=270, spheres=200, grid=50, shadow_size=512),
        # a window of no round size; shadows without ambient occlusion, so
        # the shading runs in one piece
        dict(scale, name="scale_1001x701_no_ao", width=1001, height=701, spheres=300, grid=77, shadow_size=1000,
             ao=False),
        # the full workload: 1.04 M triangles, five 2048^2 shadow maps, AO;
        # a program that shows or encodes every frame reads it into
        # page-locked memory
        dict(scale, name="scale_1080p", width=1920, height=1080),
        # the same scene for a 4K display
        dict(scale, name="scale_2160p", width=3840, height=2160),
        # data generation: 64 unlike views (256^2 to 1080p, 10k to 500k
        # triangles, 1 to 8 lights), every image kept
        dict(name="batch_64", kind="batch", views=64, min_tris=10_000, max_tris=500_000, min_px=256 * 256,
             max_px=1920 * 1080, shadow_size=1024),
        # one inverse-rendering step with a fresh frame (100k triangles)
        dict(name="adjoint_512", kind="adjoint", width=512, height=512, spheres=104),
        # new lights and materials over a frame already drawn
        dict(name="relight_640x360", kind="relight", width=640, height=360, spheres=104),
        # inverse rendering of materials and lights from 32 views, the state
        # rebuilt from the visibility at every step
        dict(name="fit_32", kind="fit", views=32, spheres=260, min_side=256, max_side=1024, shadow_size=1024, steps=20,
             stored=False, albedo=False),
        # a few views with the per-pixel state stored once
        dict(name="fit_6_stored", kind="fit", views=6, spheres=120, min_side=200, max_side=500, shadow_size=512,
             steps=20, stored=True, albedo=False),
        # and with the vertex colours among the parameters
        dict(name="fit_4_albedo", kind="fit", views=4, spheres=60, min_side=200, max_side=500, shadow_size=512,
             steps=10, stored=False, albedo=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "batch", "adjoint", "relight", "fit"])
    aspect = rng.uniform(0.75, 2.0)
    if kind == "frame":
        scene = rng.choice(["plain", "textured", "scale", "scale", "scale"])
        msaa = rng.choice([1, 1, 1, 2]) if scene != "textured" else rng.choice([1, 2, 3])
        side = math.exp(rng.uniform(math.log(64), math.log(2600 / msaa)))
        w, h = max(16, int(side * math.sqrt(aspect))), max(16, int(side / math.sqrt(aspect)))
        c = dict(kind="frame", scene=scene, width=min(w, 3840), height=min(h, 2160), msaa=msaa,
                 ao=scene != "plain" and rng.random() < 0.6, shadows=scene != "plain" and rng.random() < 0.75,
                 pinned=rng.random() < 0.5)
        if scene == "scale":
            c.update(spheres=_log_int(rng, 10, 1000), grid=_log_int(rng, 4, 200),
                     shadow_size=rng.choice([0, 512, 777, 1024, 2048]) if w * h * msaa * msaa < 1 << 20
                     else rng.choice([512, 1024, 2048]))
        return c
    if kind == "batch":
        return dict(kind="batch", views=_log_int(rng, 2, 48), min_tris=10_000, max_tris=_log_int(rng, 20_000, 500_000),
                    min_px=_log_int(rng, 64 * 64, 256 * 256), max_px=_log_int(rng, 256 * 256, 1920 * 1080),
                    shadow_size=rng.choice([512, 1000, 1024]))
    if kind in ("adjoint", "relight"):
        side = math.exp(rng.uniform(math.log(64), math.log(1100)))
        return dict(kind=kind, width=max(16, int(side * math.sqrt(aspect))),
                    height=max(16, int(side / math.sqrt(aspect))), spheres=_log_int(rng, 8, 260))
    albedo = rng.random() < 0.3
    return dict(kind="fit", views=_log_int(rng, 1, 24), spheres=_log_int(rng, 20, 260), min_side=_log_int(rng, 64, 256),
                max_side=_log_int(rng, 257, 800), shadow_size=rng.choice([512, 1000, 1024]),
                steps=rng.choice([5, 10, 20]), stored=not albedo and rng.random() < 0.5, albedo=albedo)


# ----------------------------------------------------------------- prepare
def _frame_scene(c, seed):
    if c["scene"] == "plain":
        s = scenes.c1_plain(seed=seed, width=c["width"], height=c["height"])
    elif c["scene"] == "textured":
        s = scenes.textured(seed=seed, width=c["width"], height=c["height"])
        s.shadow_map = c["shadows"]
        for light in s.lights:
            light.cast_shadow = c["shadows"]
        for m in s.materials:
            m.receive_shadow, m.ambient_occlusion = c["shadows"], c["ao"]
    else:
        s = scenes.c2_scale(seed=seed, width=c["width"], height=c["height"], n_spheres=c["spheres"], grid=c["grid"],
                            shadow_size=c["shadow_size"], ao=c["ao"], shadows=c["shadows"])
    s.msaa = c["msaa"]
    return s


def _view_sizes(n, min_px, max_px, max_aspect):
    """The image sizes of n unlike views, the same ones for every scene:
    pixels log-uniform over the range, aspect uniform."""
    rng = np.random.default_rng(n)
    sizes = []
    for _ in range(n):
        area = math.exp(rng.uniform(math.log(min_px), math.log(max_px)))
        w = max(16, int(round(math.sqrt(area * rng.uniform(0.75, max_aspect)))))
        sizes.append((w, max(16, int(round(area / w)))))
    return sizes


def _batch_scenes(c, seed):
    views = scenes.c3_views(seed=seed, n_views=c["views"], min_tris=c["min_tris"], max_tris=c["max_tris"],
                            min_px=c["min_px"], max_px=c["max_px"], shadow_size=c["shadow_size"])
    for s, (w, h) in zip(views, _view_sizes(c["views"], c["min_px"], c["max_px"], 2.0)):
        s.width, s.height = w, h
    return views


def _fit_scene(c, seed):
    s, cams = scenes.c5_inverse(seed=seed, n_views=c["views"], n_spheres=c["spheres"], min_side=c["min_side"],
                                max_side=c["max_side"], shadow_size=c["shadow_size"])
    sizes = _view_sizes(c["views"], c["min_side"] ** 2, c["max_side"] ** 2, 1.5)
    return s, [(cam, w, h) for (cam, _, _), (w, h) in zip(cams, sizes)]


def _fit_groups(c):
    return ("kd", "ks", "shininess", "light_pos", "light_int") + (("albedo",) if c["albedo"] else ())


def _start_of(truth, seed, sigma):
    return diff.perturb(truth, np.random.default_rng(seed + 1), sigma)


def prepare(case, seed):
    c, dev = case, _device()
    if c["kind"] == "frame":
        r = render.renderer_for(_frame_scene(c, seed), dev)
        host = render.pinned_array((r.H, r.W, 4)) if c["pinned"] else None
        return dict(case=c, r=r, host=host)
    if c["kind"] == "batch":
        rs = [render.renderer_for(s, dev) for s in _batch_scenes(c, seed)]
        return dict(case=c, rs=rs, hosts=[render.pinned_array((r.H, r.W, 4)) for r in rs])
    if c["kind"] in ("adjoint", "relight"):
        s = scenes.c4_adjoint(seed=seed, width=c["width"], height=c["height"], n_spheres=c["spheres"])
        r = render.renderer_for(s, dev)
        r.render_device()
        truth = diff.scene_params(s)
        start = _start_of(truth, seed, 0.1)
        # the observed image: the scene as it is; uncovered pixels count for nothing
        target = np.nan_to_num(r.ForwardLinear(truth)) if c["kind"] == "adjoint" else None
        return dict(case=c, r=r, start=start, target=target)
    s, cams = _fit_scene(c, seed)
    gs, rs = render.views_of(s, cams, dev)
    render.render_batch(rs)
    truth = diff.scene_params(s)
    fit = diff.Fit(rs, stored_gbuffer=c["stored"])
    fit.targets(truth)
    return dict(case=c, gs=gs, rs=rs, fit=fit, start=_start_of(truth, seed, 0.2))


# --------------------------------------------------------------------- run
def run(state):
    c = state["case"]
    if c["kind"] == "frame":
        if not c["pinned"]:
            return state["r"].Render()
        state["r"].render_device()
        return state["r"].image(state["host"])
    if c["kind"] == "batch":
        render.render_batch(state["rs"])
        for r, host in zip(state["rs"], state["hosts"]):
            r.image(host)
        return state["hosts"]
    if c["kind"] == "adjoint":
        state["r"].render_device()
        loss, g = state["r"].Backward(state["start"], state["target"])
        return dict(loss=loss, grads=g.arrays())
    if c["kind"] == "relight":
        return dict(linear=state["r"].ForwardLinear(state["start"]))
    p, hist = state["fit"].run(state["start"], steps=c["steps"], lr=1e-2, groups=_fit_groups(c))
    # (sums of squares of float32 differences, kept as float32 for a plot)
    return dict(params=p.arrays(), loss=hist.astype(np.float32))


# -------------------------------------------------------------------- work
SPHERE_V, SPHERE_T = 482, 960  # scenes.uv_sphere
COVERED = 0.4                  # of a frame's pixels, typically


def _frame_work(P, P_out, V, T, meshes, lights, slots, S, ao):
    """One frame.  Bytes: the scene (shared meshes at 52 bytes a vertex with
    its share of triangles, a matrix and a material base per object) in, the
    image out.  Flops: every vertex into the main view (matrix, divide,
    normal, back transform) and into every light's, every triangle's cull, box
    and area per view; per covered pixel its fragment, the lights' terms, a
    shadow lookup per map and 8 x 99 AO taps of a difference, a product and a
    maximum."""
    flops = V * (130 + 35 * slots) + T * (1 + slots) * 25
    flops += COVERED * P * (150 + lights * 90 + slots * 60 + (8 * 99 * 3 if ao else 0))
    return dict(bytes=meshes + 4 * P_out, flops=flops)


def work(case):
    c = case
    if c["kind"] == "frame":
        P_out = c["width"] * c["height"]
        P = P_out * c["msaa"] ** 2
        if c["scene"] == "scale":
            g = c["grid"]
            V, T = c["spheres"] * SPHERE_V + (g + 1) ** 2, c["spheres"] * SPHERE_T + 2 * g * g
            mesh, lights, S = (SPHERE_V + (g + 1) ** 2) * 52 + (SPHERE_T + 2 * g * g) * 16 + c["spheres"] * 72, 5, \
                c["shadow_size"]
        else:
            V, T, mesh, lights, S = SPHERE_V + 28, SPHERE_T + 16, SPHERE_V * 52 + SPHERE_T * 16, 2, 0
            if c["scene"] == "textured":
                mesh += (256 * 256 + 96 * 40) * 4 * 4 // 3
        return _frame_work(P, P_out, V, T, mesh, lights, lights if c["shadows"] else 0, S, c["ao"])
    if c["kind"] == "batch":
        # the ranges' log-uniform means
        px = (c["max_px"] - c["min_px"]) / max(1e-9, math.log(c["max_px"] / c["min_px"]))
        T = (c["max_tris"] - c["min_tris"]) / max(1e-9, math.log(c["max_tris"] / c["min_tris"]))
        w = _frame_work(px, px, T * SPHERE_V / SPHERE_T, T, SPHERE_V * 52 + SPHERE_T * 16 + T / SPHERE_T * 72, 4.5, 4.5,
                        c["shadow_size"], False)
        return {k: v * c["views"] for k, v in w.items()}
    V = c["spheres"] * SPHERE_V
    if c["kind"] == "relight":
        P = c["width"] * c["height"]
        return dict(bytes=P * (8 + 12) + 24 * V, flops=COVERED * P * (120 + 4 * 90))
    if c["kind"] == "adjoint":
        P = c["width"] * c["height"]
        w = _frame_work(P, P, V, c["spheres"] * SPHERE_T, SPHERE_V * 52 + SPHERE_T * 16 + c["spheres"] * 72, 4, 0, 0,
                        False)
        # the target in, the vertices' colours in and gradients out
        return dict(bytes=w["bytes"] + 12 * P + 36 * V, flops=w["flops"] + COVERED * P * (200 + 4 * 300))
    # per pixel its state (rebuilt from an 8-byte key and a shadow count, or
    # 52 stored bytes) and its target; per step and covered pixel the shading
    # and its adjoint
    a, b = c["min_side"] ** 2, c["max_side"] ** 2
    P = c["views"] * (b - a) / math.log(b / a)
    per_px = (52 if c["stored"] else 9) + 12
    return dict(bytes=P * per_px + (24 if c["albedo"] else 12) * V,
                flops=c["steps"] * COVERED * P * (200 + 4 * 300))


# ------------------------------------------------------------------- exact
# The differentiable shading in float64: the vertices transformed, the
# visibility and the shadow maps rasterised, the shading, its gradients by
# autograd, Adam.
F64 = torch.float64


def _t(a, dev):
    return torch.as_tensor(np.asarray(a), device=dev)


def _f32(x):
    return np.asarray(x, np.float32).astype(np.float64)


def _view_matrix(pos, target, up):
    pos, target, up = _f32(pos), _f32(target), _f32(up)
    f = (target - pos) / np.linalg.norm(target - pos)
    s = np.cross(f, up)
    s /= np.linalg.norm(s)
    u = np.cross(s, f)
    u /= np.linalg.norm(u)
    m = np.eye(4)
    m[0, :3], m[1, :3], m[2, :3] = s, u, -f
    m[0, 3], m[1, 3], m[2, 3] = -s @ pos, -u @ pos, f @ pos
    return m


def _perspective(fov, aspect, n, f):
    t = math.tan(float(_f32(fov)) * math.pi / 360)
    a, n, f = float(_f32(aspect)), float(_f32(n)), float(_f32(f))
    return np.array([[-1 / (a * t), 0, 0, 0], [0, -1 / t, 0, 0], [0, 0, (n + f) / (n - f), 2 * n * f / (n - f)],
                     [0, 0, 1, 0]])


def _viewport(w, h):
    return np.array([[w / 2, 0, 0, w / 2], [0, h / 2, 0, h / 2], [0, 0, 1, 0], [0, 0, 0, 1]], np.float64)


class _Geometry:
    """Every object's vertices and triangles, flat, in float64."""

    def __init__(self, s, dev):
        self.dev, self.s = dev, s
        model = _t(_f32(s.obj_model).reshape(-1, 4, 4), dev)
        nm = torch.linalg.inv(model).transpose(1, 2)
        pos, nor, tri, mat, base = [], [], [], [], 0
        for o, m in enumerate(s.obj_mesh):
            mesh = s.meshes[m]
            pos.append(_t(_f32(mesh.pos), dev) @ model[o].T)
            nor.append((_t(_f32(mesh.nor), dev) @ nm[o].T)[:, :3])
            tri.append(_t(mesh.tri.astype(np.int64), dev) + base)
            mat.append(_t(mesh.mat.astype(np.int64), dev) + int(s.obj_mat_base[o]))
            base += mesh.pos.shape[0]
        self.pos, self.nor, self.tri, self.mat = torch.cat(pos), torch.cat(nor), torch.cat(tri), torch.cat(mat)


def _barycentric(P, px, py):
    a, b, c = P[:, 0], P[:, 1], P[:, 2]
    area = (b[:, 0] - a[:, 0]) * (c[:, 1] - a[:, 1]) - (b[:, 1] - a[:, 1]) * (c[:, 0] - a[:, 0])
    w0 = (c[:, 0] - b[:, 0]) * (py - b[:, 1]) - (c[:, 1] - b[:, 1]) * (px - b[:, 0])
    w1 = (px - a[:, 0]) * (c[:, 1] - a[:, 1]) - (py - a[:, 1]) * (c[:, 0] - a[:, 0])
    w2 = (b[:, 0] - a[:, 0]) * (py - a[:, 1]) - (b[:, 1] - a[:, 1]) * (px - a[:, 0])
    return torch.stack([w0, w1, w2], 1) / area[:, None]


def _rasterise(scr, tri, W, H):
    """The nearest depth of every pixel (-inf: none) and the first triangle
    that has it."""
    dev = scr.device
    depth = torch.full((W * H,), -math.inf, dtype=F64, device=dev)
    first = torch.full((W * H,), tri.shape[0], dtype=torch.int64, device=dev)
    P = scr[tri]
    e1, e2 = P[:, 1] - P[:, 0], P[:, 2] - P[:, 0]
    lo, hi = P.amin(1), P.amax(1)
    x0 = torch.ceil(lo[:, 0] - 0.5 - 1e-6).clamp(0, W).long()
    y0 = torch.ceil(lo[:, 1] - 0.5 - 1e-6).clamp(0, H).long()
    x1 = torch.floor(hi[:, 0] - 0.5 + 1e-6).clamp(-1, W - 1).long()
    y1 = torch.floor(hi[:, 1] - 0.5 + 1e-6).clamp(-1, H - 1).long()
    n = (x1 - x0 + 1).clamp(min=0) * (y1 - y0 + 1).clamp(min=0)
    n[(e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0]) <= 0] = 0
    keep = torch.nonzero(n).flatten()
    n = n[keep]
    ends = torch.cumsum(n, 0)
    hits = []
    at = 0
    while at < keep.numel():  # 2^24 candidate pixels at a time
        before = int(ends[at] - n[at])
        to = max(at + 1, int(torch.searchsorted(ends, before + (1 << 24))))
        g, m = keep[at:to], n[at:to]
        own = torch.repeat_interleave(torch.arange(to - at, device=dev), m)
        k = torch.arange(own.numel(), device=dev) - (torch.cumsum(m, 0) - m)[own]
        g = g[own]
        w = x1[g] - x0[g] + 1
        x, y = x0[g] + k % w, y0[g] + k // w
        bc = _barycentric(P[g], x + 0.5, y + 0.5)
        ok = (bc >= -1e-7).all(1)
        g, o, z = g[ok], (y * W + x)[ok], (bc[ok] * P[g[ok]][:, :, 2]).sum(1)
        depth.scatter_reduce_(0, o, z, "amax")
        hits.append((g, o, z))
        at = to
    for g, o, z in hits:
        top = z == depth[o]
        first.scatter_reduce_(0, o[top], g[top], "amin")
    return depth, first


def _pixels(geo, cam, W, H):
    """The covered pixels of a view: what the shading needs of each."""
    s, dev = geo.s, geo.dev
    view = _view_matrix(cam["position"], cam.get("target", (0, 0, 0)), cam.get("up", (0, 1, 0)))
    proj = _perspective(cam["fov"], np.float32(W) / np.float32(H), cam["near"], cam["far"])
    vp = _viewport(W, H)
    vinv, pinv, vpinv = np.linalg.inv(view), np.linalg.inv(proj), np.linalg.inv(vp)
    clip = geo.pos @ _t(proj @ view, dev).T
    scr = clip @ _t(vp, dev).T
    scr = scr / scr[:, 3:]
    rw = -1 / clip[:, 3]
    back = (scr @ _t(vinv @ pinv @ vpinv, dev).T)[:, :3]  # (not divided by w, as the renderer keeps it)
    depth, first = _rasterise(scr[:, :3], geo.tri, W, H)
    o = torch.nonzero(first < geo.tri.shape[0]).flatten()
    g = first[o]
    vid = geo.tri[g]
    px, py = (o % W).to(F64), (o // W).to(F64)
    bc = _barycentric(scr[vid][:, :, :3], px + 0.5, py + 0.5)
    w = bc * rw[vid]
    w = w / w.sum(1, keepdim=True)
    x = (bc[:, :, None] * back[vid]).sum(1)
    V = torch.nn.functional.normalize(_t(_f32(cam["position"]), dev) - x, dim=1)
    count = torch.zeros(o.numel(), dtype=F64, device=dev)
    if s.shadow_map:
        q0 = torch.stack([px, py, depth[o], torch.ones_like(px)], 1) @ _t(vinv @ pinv @ vpinv, dev).T
        corners = np.array([[i, j, k, 1] for i in (-1, 1) for j in (-1, 1) for k in (-1, 1)], np.float64)
        S, svp = s.shadow_size, _viewport(s.shadow_size, s.shadow_size)
        for light in s.lights:
            lv = _view_matrix(light.position, s.center(), (0, 1, 0))
            q = corners @ (lv @ vinv @ pinv).T
            q = q[:, :3] / q[:, 3:]
            lo, hi = q.min(0), q.max(0)
            n, f = hi[2], lo[2] - 2
            lp = np.array([[2 / (hi[0] - lo[0]), 0, 0, (lo[0] + hi[0]) / (lo[0] - hi[0])],
                           [0, 2 / (hi[1] - lo[1]), 0, (lo[1] + hi[1]) / (lo[1] - hi[1])],
                           [0, 0, 2 / (n - f), (f + n) / (f - n)], [0, 0, 0, 1]])
            m = _t(svp @ lp @ lv, dev)
            smap, _ = _rasterise((geo.pos @ m.T)[:, :3], geo.tri, S, S)
            smap = smap.clamp(min=0)
            q = q0 @ m.T
            q = q / q[:, 3:]
            at = torch.trunc(q[:, 0]).long() + torch.trunc(q[:, 1]).long() * S
            inside = (at > 0) & (at < S * S)
            count += inside & (q[:, 2] < smap[at.clamp(0, S * S - 1)] - float(np.float32(0.03)))
    return dict(o=o, vid=vid, bc=bc, w=w, x=x, V=V, mat=geo.mat[g], sw=0.5 ** count)


def _shade(s, pix, p):
    """The linear shading of a view's covered pixels."""
    dev = pix["x"].device
    a = (pix["w"][:, :, None] * p["albedo"][pix["vid"]]).sum(1)
    n = torch.nn.functional.normalize((pix["bc"][:, :, None] * p["normal"][pix["vid"]]).sum(1), dim=1)
    kd, ks, shin = p["kd"][pix["mat"]], p["ks"][pix["mat"]], p["shininess"][pix["mat"]]
    sld, sls = 0.0, 0.0
    for i, light in enumerate(s.lights):  # (point lights only in these scenes)
        d = p["light_pos"][i] - pix["x"]
        dl = torch.linalg.norm(d, dim=1, keepdim=True)
        L = d / dl
        I = p["light_int"][i] / dl
        h = torch.nn.functional.normalize(L + pix["V"], dim=1)
        ld = (n * L).sum(1, keepdim=True).clamp(0, 1)
        ls = (n * h).sum(1).clamp(0, 1).pow(shin)[:, None]
        sld = sld + ld * I
        sls = sls + ls * I * _t(_f32(light.color[:3]), dev)
    ambient = float(sum(np.float32(e) for e in s.ambient))
    return pix["sw"][:, None] * (ambient * a + kd * sld * a / 255 + ks * sls / 255)


def _params64(p, geo):
    t = {n: _t(np.asarray(getattr(p, n), np.float64), geo.dev) for n in diff.DiffParams.NAMES if n != "normal"}
    return dict(t, normal=geo.nor)


def exact(case, seed):
    c = case
    if c["kind"] in ("frame", "batch"):
        return None  # 8-bit images
    dev = "cuda:0" if torch.cuda.is_available() else "cpu"
    if c["kind"] != "fit":
        s = scenes.c4_adjoint(seed=seed, width=c["width"], height=c["height"], n_spheres=c["spheres"])
        geo = _Geometry(s, dev)
        pix = _pixels(geo, s.camera, c["width"], c["height"])
        truth = diff.scene_params(s)
        p = _params64(_start_of(truth, seed, 0.1), geo)
        if c["kind"] == "relight":
            lin = torch.full((c["height"] * c["width"], 3), math.nan, dtype=F64, device=dev)
            lin[pix["o"]] = _shade(s, pix, p)
            return dict(linear=lin.view(c["height"], c["width"], 3).cpu().numpy())
        target = _shade(s, pix, _params64(truth, geo))
        for v in p.values():
            v.requires_grad_(True)
        loss = (_shade(s, pix, p) - target).square().sum()
        loss.backward()
        return dict(loss=float(loss.detach()), grads={n: p[n].grad.cpu().numpy() for n in diff.DiffParams.NAMES})
    s, cams = _fit_scene(c, seed)
    truth = diff.scene_params(s)
    geo = _Geometry(s, dev)
    views = [_pixels(geo, cam, w, h) for cam, w, h in cams]
    with torch.no_grad():
        t = _params64(truth, geo)
        targets = [_shade(s, v, t) for v in views]
    base = _params64(_start_of(truth, seed, 0.2), geo)
    groups = _fit_groups(c)
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    lr, eps = float(np.float32(1e-2)), float(np.float32(1e-8))
    par = {n: v.clone() for n, v in base.items()}
    theta, m, v2 = ({n: torch.zeros_like(base[n]) for n in groups} for _ in range(3))
    hist = []
    for k in range(1, c["steps"] + 1):
        for n in groups:
            par[n] = par[n].detach().requires_grad_(True)
        loss = 0.0
        for pix, target in zip(views, targets):
            part = (_shade(s, pix, par) - target).square().sum()
            part.backward()
            loss += float(part.detach())
        hist.append(loss)
        with torch.no_grad():
            for n in groups:
                g = par[n].grad * base[n]
                m[n] = b1 * m[n] + (1 - b1) * g
                v2[n] = b2 * v2[n] + (1 - b2) * g * g
                theta[n] = theta[n] - lr * (m[n] / (1 - b1 ** k)) / ((v2[n] / (1 - b2 ** k)).sqrt() + eps)
                new = base[n] * (1 + theta[n])
                if n != "light_pos":
                    theta[n] = torch.where((new < 0) & (base[n] != 0), torch.full_like(new, -1.0), theta[n])
                    new = new.clamp(min=0)
                par[n] = new
    return dict(params={n: par[n].detach().cpu().numpy() for n in diff.DiffParams.NAMES if n != "normal"},
                loss=np.array(hist))
