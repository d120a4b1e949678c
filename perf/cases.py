"""Performance cases of the framework: what its users have it do, through the public entry points.

A case is one call pattern at one size; listed() names twelve, draw() gives more
of the same ranges.  Scenes are the repository's procedural ones (Cornell box,
sphere grid, fBm heightfield under the HDR environment).  A scene and, where a
program renders one image after another, its renderer are built once per
process and kept, as such a program keeps them; a case's inputs (camera, path
seed, rays, images, weights, training data) come from the seed alone.

torch is imported before the library, which then shares torch's HIP runtime:
rays, images and training data are torch tensors handed over by pointer.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import cudapt_amd as ca
from cudapt_amd import learned, scenes

MODES = {"bdpt": ca.CPT_MODE_BDPT_STREAM, "pll": ca.CPT_MODE_BDPT_ADAPTIVE_PLL,
         "binary": ca.CPT_MODE_BDPT_ADAPTIVE_BINARY, "emp": ca.CPT_MODE_BDPT_ADAPTIVE_EMP,
         "pt": ca.CPT_MODE_PT_STREAM, "disney": ca.CPT_MODE_PT_DISNEY_MIS}
VIEW_SIZES = ((256, 256), (640, 480), (1280, 720), (333, 187))   # of the multi-view batch, in turn
HIDDEN, INPUTS = ca.MLP_HIDDEN, ca.MLP_INPUTS


def listed():
    return [
        # a viewer that refines a small scene: one Render call per frame at the parity image's size
        {"name": "frame_cornell_256", "kind": "frame", "scene": "cornell", "width": 256, "height": 256, "depth": 5},
        # the reference application's window: one Render call per frame at 800 x 600 on a full scene
        {"name": "frame_grid_800x600", "kind": "frame", "scene": "grid", "width": 800, "height": 600, "depth": 5},
        # a still: the headline render, 64 samples per pixel in one call
        {"name": "still_grid_1280x720", "kind": "still", "scene": "grid", "mode": "bdpt", "width": 1280,
         "height": 720, "depth": 8, "frames": 64},
        # learned adaptive rendering: the frames it needs to reach plain adaptive sampling's error
        {"name": "learned_field_1920x1080", "kind": "adaptive", "scene": "field", "mode": "pll", "learned": True,
         "width": 1920, "height": 1080, "depth": 8, "frames": 12},
        # the reference's own method (filter residual, bisected acceptance rounds) at its window size
        {"name": "binary_grid_800x600", "kind": "adaptive", "scene": "grid", "mode": "binary", "learned": False,
         "width": 800, "height": 600, "depth": 5, "frames": 16},
        # a data set of views: eight cameras of uneven resolution traced as one wavefront
        {"name": "views_field_8", "kind": "views", "scene": "field", "views": 8, "frames": 8, "in_flight": 6,
         "depth": 8},
        # a ray-casting service: closest hits of rays held in device memory (camera rays and scattered ones)
        {"name": "closest_grid_2m", "kind": "closest", "scene": "grid", "rays": 2097143, "layout": 0},
        # a picking query: a few host rays in, hits out
        {"name": "closest_cornell_host", "kind": "closest_host", "scene": "cornell", "rays": 1021},
        # visibility between surface points: device rays in, flags out
        {"name": "occluded_field_1m", "kind": "occluded", "scene": "field", "rays": 1000003},
        # denoising a full-HD frame with the albedo guide
        {"name": "filter_1920x1080", "kind": "filter", "width": 1920, "height": 1080, "radius": 5, "diff": True},
        # training the error model: a run of Adam steps over a device data set, between two loss readings
        {"name": "mlp_train_65536", "kind": "mlp_train", "batch": 65536, "steps": 32},
        # the model on every pixel of a full-HD frame
        {"name": "mlp_infer_2m", "kind": "mlp_infer", "n": 1920 * 1080},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "still", "adaptive", "views", "closest", "closest_host", "occluded", "filter",
                       "mlp_train", "mlp_infer"])
    c = {"kind": kind}
    if kind == "frame":
        w = _log(rng, 96, 1280)
        c.update(scene=rng.choice(["cornell", "grid", "small_grid"]), width=w, height=max(54, w * 9 // 16 + rng.randint(0, 9)),
                 depth=rng.randint(3, 8))
    elif kind == "still":
        w = _log(rng, 200, 1280)
        c.update(scene=rng.choice(["cornell", "grid", "small_grid"]), mode=rng.choice(["bdpt", "bdpt", "pt", "disney"]),
                 width=w, height=w * 9 // 16, depth=rng.randint(3, 8), frames=_log(rng, 3, 48))
    elif kind == "adaptive":
        w = _log(rng, 320, 1600)
        mode = rng.choice(["pll", "pll", "binary", "emp"])
        c.update(scene=rng.choice(["grid", "field"]), mode=mode, learned=mode == "pll" and rng.random() < 0.5, width=w,
                 height=w * 9 // 16 + rng.randint(0, 5), depth=rng.randint(4, 8), frames=rng.randint(7, 14))
    elif kind == "views":
        c.update(scene=rng.choice(["grid", "field"]), views=rng.randint(2, 8), frames=rng.randint(2, 8),
                 in_flight=rng.randint(1, 6), depth=rng.randint(4, 8))
    elif kind == "closest":
        c.update(scene=rng.choice(["cornell", "grid", "field"]), rays=_log(rng, 4000, 2000000),
                 layout=rng.choice([0, 2]))
    elif kind == "closest_host":
        c.update(scene=rng.choice(["cornell", "grid", "field"]), rays=_log(rng, 100, 100000))
    elif kind == "occluded":
        c.update(scene=rng.choice(["cornell", "grid", "field"]), rays=_log(rng, 4000, 2000000))
    elif kind == "filter":
        w = _log(rng, 200, 1920)
        c.update(width=w, height=w * 9 // 16 + rng.randint(0, 7), radius=rng.randint(1, 9), diff=rng.random() < 0.5)
    elif kind == "mlp_train":
        c.update(batch=_log(rng, 500, 65536), steps=rng.randint(4, 32))
    else:
        c.update(n=_log(rng, 1000, 2000000))
    return c


# ---- scenes and renderers, built once per process ----------------------------

@functools.lru_cache(maxsize=4)
def _scene(name):
    if name == "cornell":
        sc = scenes.cornell()
    elif name == "grid":
        sc = scenes.sphere_grid()                       # 262,306 triangles
    elif name == "small_grid":
        sc = scenes.sphere_grid(grid=16)                # 16,546 triangles
    else:
        sc = scenes.heightfield(light="env")            # 1,050,976 triangles
    return sc, ca.Scene(sc)


@functools.lru_cache(maxsize=1)
def _renderer(mode, width, height, depth, frames, field):
    """The renderer that a program keeps while cameras change."""
    attribs = {"eye_depth": depth}
    if mode in ("bdpt", "pll", "binary", "emp"):
        attribs["light_depth"] = depth
    if field and mode in ("pll", "binary"):
        attribs.update(scenes.ADAPTIVE_C3)
    if mode == "pll":
        attribs["Learned Signal"] = 3                   # as the learned protocol runs: with the filter residual
    if mode in ("bdpt", "pt", "disney"):
        attribs["Frames In Flight"] = min(frames, 64)
    return ca.Renderer(width, height, mode=MODES[mode], **attribs)


def _camera(scene, seed, width=16, height=9):
    """A view of the scene: the heightfield's seeded poses, the others' own camera moved a little."""
    if scene == "field":
        return learned.heightfield_poses(1, seed0=0xCA3E0000 + seed % 100003, width=width, height=height)[0]
    cam = dict(_scene(scene)[0]["camera"])
    step = 0.02 if scene == "cornell" else 1.0
    r = np.random.default_rng(seed)
    cam["pos"] = tuple(float(p + step * r.uniform(-1, 1)) for p in cam["pos"])
    return cam


def _weights(rng):
    """Glorot-uniform weights and small biases of the 9-64-64-1 model, one flat vector."""
    def glorot(i, o):
        return rng.uniform(-1, 1, i * o) * math.sqrt(6.0 / (i + o))
    return np.concatenate([glorot(INPUTS, HIDDEN), rng.normal(0, 0.05, HIDDEN), glorot(HIDDEN, HIDDEN),
                           rng.normal(0, 0.05, HIDDEN), glorot(HIDDEN, 1), rng.normal(0, 0.05, 1)]).astype(np.float32)


class _Array:
    """A torch tensor where the API takes a DeviceBuffer (pointer and size)."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _camera_rays(cam, n, g):
    """n pinhole rays of a 16:9 image in pixel order, jittered."""
    h = max(1, int(math.sqrt(n * 9 / 16)))
    w = -(-n // h)
    i = torch.arange(n, device="cuda")
    x, y = (i % w).float() + torch.rand(n, device="cuda", generator=g), (i // w).float() + torch.rand(n, device="cuda", generator=g)
    d = np.asarray(cam["dir"], np.float64)
    right = np.cross(d, cam["up"])
    right /= np.linalg.norm(right)
    up = np.cross(right, d)
    tf = math.tan(cam["fov"] / 2)
    u, v = ((2 * x / w - 1) * tf * w / h)[:, None], ((2 * y / h - 1) * tf)[:, None]
    t = lambda a: torch.tensor(np.asarray(a, np.float32), device="cuda")[None]  # noqa: E731
    dirs = t(right) * u + t(up) * v + t(d)
    return t(cam["pos"]).expand(n, 3), dirs / dirs.norm(dim=1, keepdim=True)


def _rays(scene, n, seed, reach):
    """n rays: the first half a camera's, in pixel order, the rest from points spread over the scene (in
    the order of a coarse grid, as paths that left neighbouring pixels are) in any direction; reach: the
    segments end within it."""
    g = _gen(seed)
    pos = _scene(scene)[0]["pos"]
    lo, hi = (torch.tensor(np.asarray(f(np.asarray(pos), 0), np.float32), device="cuda") for f in (np.min, np.max))
    k = n // 2
    o1, d1 = _camera_rays(_camera(scene, seed), k, g)
    m = n - k
    o2 = lo + (hi - lo) * torch.rand(m, 3, device="cuda", generator=g)
    cell = ((o2 - lo) / (hi - lo) * 15.99).long()
    o2 = o2[torch.argsort((cell[:, 2] * 16 + cell[:, 0]) * 16 + cell[:, 1])]
    d2 = torch.randn(m, 3, device="cuda", generator=g)
    d2 = d2 / d2.norm(dim=1, keepdim=True)
    r = torch.empty(n, 8, device="cuda")
    r[:k, 0:3], r[k:, 0:3], r[:k, 4:7], r[k:, 4:7] = o1, o2, d1, d2
    r[:, 3], r[:, 7] = 1e20, 1e-4
    if reach:
        r[:, 3] = float((hi - lo).max()) * (0.02 + 0.5 * torch.rand(n, device="cuda", generator=g))
    return r


def _image(c, seed):
    """Guides and a noisy image as an adaptive frame leaves them: a rolling ground with boxes on it."""
    W, H, g = c["width"], c["height"], _gen(seed)
    y, x = torch.meshgrid(torch.arange(H, device="cuda").float(), torch.arange(W, device="cuda").float(), indexing="ij")
    ph = torch.rand(8, device="cuda", generator=g) * 6.283
    z = 20 + 0.01 * y + 0.8 * torch.sin(x * 0.021 + ph[0]) + 0.5 * torch.cos(y * 0.033 + ph[1])
    block = ((x * 0.013 + ph[2]).floor() * 7 + (y * 0.017 + ph[3]).floor() * 13) % 5
    z = z - block
    pos = torch.stack([(x - W / 2) * z / W, (y - H / 2) * z / W, z], -1)
    nrm = torch.stack([0.3 * torch.cos(x * 0.021 + ph[0]), 0.2 * torch.sin(y * 0.033 + ph[1]), torch.ones_like(x)], -1)
    nrm = nrm / nrm.norm(dim=-1, keepdim=True)
    diff = torch.stack([0.2 + 0.12 * block, 0.7 - 0.1 * block, 0.3 + 0.05 * block], -1)
    light = (0.4 + 0.6 * nrm[..., :1] ** 2)
    n = torch.randint(1, 60, (H, W), device="cuda", generator=g, dtype=torch.int32)
    col = diff * light * (1 + torch.randn(H, W, 3, device="cuda", generator=g) / n[..., None].float().sqrt()).clamp_min(0)
    return [t.contiguous() for t in (col, pos, nrm, diff)], n


SIGMAS = (50.0, 1.0, 0.25, 0.1)          # colour, position, normal, albedo: the adaptive renderer's defaults
ND = 5


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "frame":
        S = _scene(c["scene"])[1]
        R = ca.Renderer(c["width"], c["height"], eye_depth=c["depth"], light_depth=c["depth"], seed=seed % 65521)
        cam = _camera(c["scene"], seed)
        R.render(S, cam, frames=1, result=False)          # the viewer's first frame: buffers exist from here on
        return {"kind": kind, "S": S, "R": R, "cam": cam}
    if kind in ("still", "adaptive"):
        S = _scene(c["scene"])[1]
        R = _renderer(c["mode"], c["width"], c["height"], c["depth"], c["frames"], c["scene"] == "field")
        s = {"kind": kind, "S": S, "R": R, "cam": _camera(c["scene"], seed, c["width"], c["height"]),
             "frames": c["frames"], "model": None}
        if c.get("learned"):
            s["model"] = ca.Mlp()
            s["model"].set_params(_weights(np.random.default_rng(seed)))
        return s
    if kind == "views":
        S = _scene(c["scene"])[1]
        views = []
        for i in range(c["views"]):
            w, h = VIEW_SIZES[i % len(VIEW_SIZES)]
            views.append(dict(_camera(c["scene"], seed + 7919 * i, w, h), width=w, height=h))
        B = ca.Batch(views, frames_in_flight=c["in_flight"], eye_depth=c["depth"], light_depth=c["depth"])
        return {"kind": kind, "S": S, "B": B, "frames": c["frames"]}
    if kind in ("closest", "occluded"):
        r = _rays(c["scene"], c["rays"], seed, kind == "occluded")
        out = torch.empty(c["rays"], 4 if kind == "closest" else 1, dtype=torch.int32, device="cuda")
        return {"kind": kind, "S": _scene(c["scene"])[1], "rays": r, "out": out, "layout": c.get("layout", 0)}
    if kind == "closest_host":
        return {"kind": kind, "S": _scene(c["scene"])[1], "rays": _rays(c["scene"], c["rays"], seed, False).cpu().numpy()}
    if kind == "filter":
        img, n = _image(c, seed)
        return {"kind": kind, "img": img, "n": n, "c": c, "out": torch.empty_like(img[0]),
                "err": torch.empty(c["height"], c["width"], device="cuda")}
    if kind == "mlp_train":
        m = ca.Mlp()
        x, t, w = _samples(c, seed)
        m.set_params(w)
        return {"kind": kind, "m": m, "x": _Array(x), "t": _Array(t), "c": c}
    m = ca.Mlp()
    x, _, w = _samples({"batch": c["n"], "steps": 1}, seed)
    m.set_params(w)
    return {"kind": kind, "m": m, "x": _Array(x), "y": _Array(torch.empty(c["n"], device="cuda")), "n": c["n"]}


def _samples(c, seed):
    """Features of the model's range, log-variance targets that depend on them, and weights."""
    g = _gen(seed)
    n = c["batch"] * min(c["steps"], 8)                   # the run's batches, gone through again after the eighth
    x = torch.randn(n, INPUTS, device="cuda", generator=g) * 0.5
    t = -4 + 2 * x[:, 0] - x[:, 3] * x[:, 5] + 0.5 * torch.randn(n, device="cuda", generator=g)
    return x.contiguous(), t.contiguous(), _weights(np.random.default_rng(seed))


def run(s):
    kind = s["kind"]
    if kind == "frame":
        return s["R"].render(s["S"], s["cam"], frames=1)
    if kind in ("still", "adaptive"):
        R = s["R"]
        if kind == "adaptive" and getattr(R, "_mlp", None) is not s["model"]:
            R.set_mlp(s["model"])
        R.reset()                                         # a new image
        return R.render(s["S"], s["cam"], frames=s["frames"])
    if kind == "views":
        B = s["B"]
        B.reset()
        B.render(s["S"], s["frames"])
        return [B.result(v) for v in range(len(B.views))]
    if kind == "closest":
        o = s["out"]
        s["S"].trace_device(s["rays"].data_ptr(), len(o), o.data_ptr(), layout=s["layout"])
        f = o.view(torch.float32)
        return {"tri": o[:, 0], "t": f[:, 1], "uv": f[:, 2:]}
    if kind == "occluded":
        o = s["out"]
        s["S"].occluded_device(s["rays"].data_ptr(), len(o), o.data_ptr())
        return o
    if kind == "closest_host":
        h = s["S"].trace(s["rays"])
        return {"tri": h["tri"], "t": h["t"], "u": h["u"], "v": h["v"]}
    if kind == "filter":
        c, p = s["c"], lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        col, pos, nrm, diff = s["img"]
        ca._check(ca.lib().cpt_filter_cross_bilateral_device(
            p(col), p(pos), p(nrm), p(diff) if c["diff"] else None, c["width"], c["height"], *SIGMAS, c["radius"],
            p(s["n"]), ND, p(s["out"]), p(s["err"]), None), "cpt_filter_cross_bilateral_device")
        return {"filtered": s["out"], "error": s["err"]}
    if kind == "mlp_train":
        c = s["c"]
        loss = s["m"].train_steps_device(s["x"], s["t"], len(s["t"].t), c["batch"], c["steps"], lr=1e-3, want_loss=True)
        return {"params": s["m"].params(), "loss": loss}
    s["m"].infer_device(s["x"], s["n"], s["y"])
    return s["y"].t


# ---- what a pass cannot do without -------------------------------------------

TRIS = {"cornell": 36, "grid": 262306, "small_grid": 16546, "field": 1050976}
# a ray: about ten 4-wide nodes (four box tests of 13 operations) and four triangle tests of 45
RAY_FLOPS = 10 * 4 * 13 + 4 * 45
# a path of the scenes: about two extension rays and half an occlusion ray, 300 operations of shading a vertex
PATH_FLOPS = 2.5 * RAY_FLOPS + 2 * 300


def work(case):
    c, kind = case, case["kind"]
    scene = TRIS.get(c.get("scene"), 0) * (36 + 36 + 4)   # triangle corners, normals and material index once
    px = c.get("width", 0) * c.get("height", 0)
    if kind in ("frame", "still"):
        return {"bytes": scene + 12 * px, "flops": float(px * c.get("frames", 1) * PATH_FLOPS)}
    if kind == "adaptive":                                # a filter pass over 121 taps beside the paths
        return {"bytes": scene + 12 * px, "flops": float(px * c["frames"] * (PATH_FLOPS + 121 * 30))}
    if kind == "views":
        px = sum(w * h for w, h in (VIEW_SIZES[i % len(VIEW_SIZES)] for i in range(c["views"])))
        return {"bytes": scene + 12 * px, "flops": float(px * c["frames"] * PATH_FLOPS)}
    if kind in ("closest", "closest_host", "occluded"):
        return {"bytes": scene + c["rays"] * (32 + (4 if kind == "occluded" else 16)), "flops": float(c["rays"] * RAY_FLOPS)}
    if kind == "filter":
        taps = (2 * c["radius"] + 1) ** 2
        return {"bytes": px * (36 + (12 if c["diff"] else 0) + 4 + 16), "flops": float(px * taps * (34 if c["diff"] else 27))}
    flop = 2 * (INPUTS * HIDDEN + HIDDEN * HIDDEN + HIDDEN)
    if kind == "mlp_train":
        n = c["batch"] * c["steps"]
        return {"bytes": c["batch"] * min(c["steps"], 8) * 40 + ca.MLP_PARAMS * 24, "flops": float(3 * flop * n)}
    return {"bytes": c["n"] * 40 + ca.MLP_PARAMS * 4, "flops": float(flop * c["n"])}


# ---- 64-bit results ----------------------------------------------------------

def _split(p):
    at, out = 0, []
    for shape in ((INPUTS, HIDDEN), (HIDDEN,), (HIDDEN, HIDDEN), (HIDDEN,), (HIDDEN, 1), (1,)):
        n = math.prod(shape)
        out.append(p[at:at + n].reshape(shape))
        at += n
    return out


def _model(p, x):
    w1, b1, w2, b2, w3, b3 = _split(p)
    gelu = functools.partial(torch.nn.functional.gelu, approximate="tanh")
    return (gelu(gelu(x @ w1 + b1) @ w2 + b2) @ w3 + b3)[:, 0]


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "mlp_infer":
        x, _, w = _samples({"batch": c["n"], "steps": 1}, seed)
        p = torch.tensor(w, device="cuda").double()
        return torch.cat([_model(p, b.double()) for b in x.split(1 << 18)])
    if kind == "mlp_train":
        x, t, w = _samples(c, seed)
        p = torch.tensor(w, device="cuda").double().requires_grad_()
        m, v, nb, B, loss = torch.zeros_like(p.detach()), torch.zeros_like(p.detach()), len(t) // c["batch"], c["batch"], None
        for k in range(c["steps"]):
            j = k % nb * B
            loss = ((_model(p, x[j:j + B].double()) - t[j:j + B].double()) ** 2).mean()
            g, = torch.autograd.grad(loss, p)
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            step = 1e-3 * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
            p = (p.detach() - step).requires_grad_()
        return {"params": p.detach(), "loss": float(loss.detach())}
    if kind == "filter":
        img, n = _image(c, seed)
        col, pos, nrm, diff = (t.double() for t in img)
        H, W, R = c["height"], c["width"], c["radius"]
        num, den = torch.zeros_like(col), torch.zeros(H, W, 1, dtype=torch.float64, device="cuda")
        ix, iy = torch.arange(W, device="cuda"), torch.arange(H, device="cuda")
        far = lambda i, n: torch.where((i < 0) | (i >= n), torch.full_like(i, n - 1), i)  # noqa: E731  off the image: the high edge
        for i in range(-R, R + 1):
            for j in range(-R, R + 1):
                at = (far(iy + i, H)[:, None], far(ix + j, W)[None])
                a = sum((((t[at] - t) ** 2).sum(-1, keepdim=True) / (2 * s * s)
                         for t, s in zip((col, pos, nrm, diff)[:4 if c["diff"] else 3], SIGMAS)))
                f = torch.exp(-a - (i * i + j * j) / (2 * SIGMAS[0] ** 2))
                num += f * col[at]
                den += f
        out = num / den
        red = ND / (ND + n.double())
        return {"filtered": out, "error": red * ((out - col) ** 2).sum(-1) / 3}
    if kind == "closest_host" and c["scene"] == "cornell":
        r = _rays("cornell", c["rays"], seed, False).double().cpu().numpy()
        sc = _scene("cornell")[0]
        p = np.asarray(sc["pos"], np.float64)[np.asarray(sc["idx"])]
        o, d = r[:, None, 0:3] + r[:, None, 7:8] * r[:, None, 4:7], r[:, None, 4:7]
        e0, e1 = (p[:, 1] - p[:, 0])[None], (p[:, 2] - p[:, 0])[None]
        q = np.cross(d, e1)
        with np.errstate(divide="ignore", invalid="ignore"):
            inv = 1.0 / (q * e0).sum(-1)
            s = o - p[None, :, 0]
            w = np.cross(s, e0)
            t, u, v = (w * e1).sum(-1) * inv, (q * s).sum(-1) * inv, (w * d).sum(-1) * inv
            ok = (np.abs(1 / inv) >= 1e-9) & (t >= 0) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1)
        t = np.where(ok, t, np.inf)
        at = t.argmin(1)
        hit = np.isfinite(t.min(1))
        pick = lambda a: np.where(hit, np.take_along_axis(np.where(ok, a, 0.0), at[:, None], 1)[:, 0], 0.0)  # noqa: E731
        return {"tri": None, "t": np.where(hit, t.min(1), np.float64(np.float32(1e20))), "u": pick(u), "v": pick(v)}
    return None                                           # paths and large scenes: no plain 64-bit form within seconds
