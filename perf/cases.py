"""Performance cases of the renderer and the denoiser: what a program that uses
this package has it do, through ``MdwtRenderer`` and ``Denoiser``.

Every case is a dict of plain values. ``kind`` says what a pass is:

* ``view``   an interactive viewer's step: one change (the camera, or one
             channel's opacity slider), one frame, the RGBA8 frame buffer read;
* ``frames`` an offline render: a fresh accumulation of ``frames`` frames, the
             float image read back (and its second moment and the denoiser's
             auxiliary buffers where they are on);
* ``batch``  many cameras of uneven size and sample count over one volume;
* ``infer``  the denoiser on one image;
* ``train``  one optimiser step of the denoiser, updated weights read back;
* ``grad``   the loss gradient of one pair.

Volumes are fractal value noise plus Gaussian blobs and the transfer functions
piecewise linear with a transparent low end, as in ``mdwtracker_amd.scenes``;
they are generated on the GPU and handed over as host arrays.
"""
from __future__ import annotations

import colorsys
import math

import numpy as np
import torch

from mdwtracker_amd.capi import MdwtRenderer
from mdwtracker_amd.denoise import Denoiser, input_width

_BYTES = {"u8": 1, "u16": 2, "f16": 2, "f32": 4}


def _render(name, kind, mode, c, dims, dtype, mc, w, h, **more):
    d = {"kind": kind, "mode": mode, "channels": c, "nx": dims[0], "ny": dims[1], "nz": dims[2],
         "dtype": dtype, "cell": mc, "width": w, "height": h, "spp": 1, "frames": 1,
         "moments": False, "aov": False, "gradient": False, "shadows": False, "edit": False}
    d.update(more)
    if name:
        d["name"] = name
    return d


def listed():
    return [
        # the smallest call: a thumbnail viewer of two small channels; launches and host work
        _render("view_small_m0", "view", 0, 2, (64, 64, 64), "u8", 8, 256, 256),
        # orbiting the camera around the 4-channel workload at full size
        _render("view_m2", "view", 2, 4, (256, 256, 256), "u8", 16, 1024, 1024),
        # dragging an opacity slider: majorants rebuilt, then a frame; odd sizes everywhere,
        # the default macrocells of 4 voxels
        _render("edit_m3_odd", "view", 3, 3, (181, 150, 133), "u16", 4, 801, 603, edit=True),
        # offline render of the 4-channel workload (the benchmark's scene and method)
        _render("frames_m2", "frames", 2, 4, (256, 256, 256), "u8", 16, 1024, 1024, frames=64),
        # several samples per pixel and frame, half-precision voxels, confidence intervals
        _render("frames_m0_spp", "frames", 0, 4, (200, 160, 120), "f16", 8, 640, 480, spp=4,
                frames=8, moments=True),
        # many float channels of a flat simulation domain
        _render("frames_m1_10ch", "frames", 1, 10, (256, 256, 64), "f32", 16, 1024, 1024, frames=8),
        # publication images: gradient shading and shadow rays
        _render("lit_m2", "frames", 2, 4, (256, 256, 256), "u8", 16, 1024, 1024, frames=8,
                gradient=True, shadows=True),
        # the ray marcher that users compare the tracking modes with
        _render("march_m8", "frames", 8, 4, (128, 128, 128), "u8", 16, 640, 480, frames=4),
        # inputs of the denoiser: image, second moment and auxiliary buffers
        _render("aov_m2", "frames", 2, 4, (192, 192, 192), "u8", 16, 512, 512, frames=64,
                moments=True, aov=True),
        # a turntable / data-set generation job: many cameras over one volume
        _render("batch_24", "batch", 2, 4, (128, 128, 128), "f16", 16, 512, 512, frames=4,
                views=24, launch=1, spp=4),
        # denoising one full-size render
        {"name": "infer_1024", "kind": "infer", "channels": 4, "width": 1024, "height": 1024},
        # training on the package's default tile and batch size
        {"name": "train_8x256", "kind": "train", "channels": 4, "width": 256, "height": 256,
         "batch": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges."""
    kind = rng.choice(["view", "view", "frames", "frames", "frames", "frames", "batch", "infer",
                       "train", "grad"])
    if kind in ("infer", "train", "grad"):
        hi = 1024 if kind == "infer" else 256
        c = {"kind": kind, "channels": rng.choice([1, 2, 4, 4, 7, 10]),
             "width": 4 * _log(rng, 16, hi // 4), "height": 4 * _log(rng, 16, hi // 4)}
        if kind == "train":
            c["batch"] = rng.randint(1, 8)
        return c
    dtype = rng.choice(["u8", "u16", "f16", "f32"])
    channels = rng.choice([1, 2, 3, 4, 4, 5, 10])
    dims = tuple(_log(rng, 48, 200) for _ in range(3))
    cell = rng.choice([4, 8, 16])
    w, h = _log(rng, 128, 1024), _log(rng, 128, 1024)
    if kind == "view":
        return _render(None, kind, rng.choice([0, 1, 2, 3, 4, 5]), channels, dims, dtype, cell, w, h,
                       edit=rng.random() < 0.5)
    if kind == "batch":
        return _render(None, kind, rng.choice([0, 2, 2, 3]), min(channels, 4), dims, dtype, cell,
                       512, 512, frames=rng.randint(1, 4), views=_log(rng, 4, 24),
                       launch=rng.choice([0, 1, 2]), spp=rng.choice([1, 2, 4]))
    what = rng.choice(["plain", "plain", "lit", "march", "aov"])
    if what == "march":
        return _render(None, kind, rng.choice([6, 7, 8]), min(channels, 4),
                       tuple(min(d, 128) for d in dims), dtype, cell, min(w, 640), min(h, 480),
                       frames=_log(rng, 1, 4))
    mode = rng.choice([0, 1, 2, 3, 4, 5])
    if what == "lit":
        return _render(None, kind, mode, min(channels, 4), dims, dtype, cell, w, h,
                       frames=_log(rng, 1, 8), gradient=rng.random() < 0.7,
                       shadows=rng.random() < 0.7)
    if what == "aov":
        return _render(None, kind, mode, min(channels, 4), dims, dtype, cell, min(w, 640),
                       min(h, 640), frames=_log(rng, 4, 64), moments=True, aov=True)
    return _render(None, kind, mode, channels, dims, dtype, cell, w, h, spp=rng.choice([1, 1, 2, 4]),
                   frames=_log(rng, 1, 16), moments=rng.random() < 0.3)


# ------------------------------------------------------------------ inputs --
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _axis(lat, n, freq, axis):
    u = (torch.arange(n, device=lat.device, dtype=torch.float32) + 0.5) / n * freq
    i = u.floor().long().clamp_(max=freq - 1)
    t = u - i
    shape = [1, 1, 1]
    shape[axis] = n
    w = (t * t * (3.0 - 2.0 * t)).view(shape)
    a, b = lat.index_select(axis, i), lat.index_select(axis, i + 1)
    return a + w * (b - a)


def _volumes(case, rng):
    """The channels as host arrays (nz, ny, nx), deterministic in rng's seed."""
    dev = _device()
    shape = (case["nz"], case["ny"], case["nx"])
    grids = [((torch.arange(n, device=dev, dtype=torch.float32) + 0.5) / n) for n in shape]
    out = []
    for _ in range(case["channels"]):
        v = torch.zeros(shape, device=dev)
        for o in range(5):
            f = 4 * 2 ** o
            lat = torch.from_numpy(rng.random((f + 1, f + 1, f + 1), np.float32)).to(dev)
            v += 0.5 ** o * _axis(_axis(_axis(lat, shape[2], f, 2), shape[1], f, 1), shape[0], f, 0)
        v /= 1.9375
        for _ in range(16):
            c, s, a = rng.uniform(0, 1, 3), rng.uniform(0.05, 0.2), rng.uniform(0.3, 1.0)
            g = [torch.exp(-((x - float(c[k])) ** 2) / (2 * s * s)) for k, x in enumerate(grids)]
            v += float(a) * g[0][:, None, None] * (g[1][:, None] * g[2][None, :])[None]
        v = (v / v.max()).clamp_(0, 1).cpu().numpy()
        t = case["dtype"]
        out.append(np.rint(255 * v).astype(np.uint8) if t == "u8" else
                   np.rint(65535 * v).astype(np.uint16) if t == "u16" else
                   v.astype(np.float16 if t == "f16" else np.float32))
    return out


def _tfs(case, rng):
    u = (np.arange(256) + 0.5) / 256
    out = []
    for c in range(case["channels"]):
        al = rng.uniform(0.0, 1.0, 8)
        al[0] = 0.0
        t = np.empty((256, 4), np.float32)
        t[:, :3] = colorsys.hsv_to_rgb(c / case["channels"], 0.8, 1.0)
        t[:, 3] = np.interp(u, np.sort(rng.uniform(0.2, 1.0, 8)), al)
        out.append(t)
    return out


def _opacity(case):
    # a step is half a voxel, so the optical depth of a voxel is 2 alpha^3 times this
    return 2.56 / max(case["nx"], case["ny"], case["nz"])


def _orbit(angle, radius=1.8, tilt=0.3):
    d = np.array([math.sin(angle), tilt, math.cos(angle)])
    d = radius * d / np.linalg.norm(d)
    return tuple(float(0.5 + x) for x in d), (0.5, 0.5, 0.5), (0.0, 1.0, 0.0), 45.0


def _camera(case, seed):
    return _orbit(float(np.random.default_rng([seed, 2]).uniform(0, 2 * math.pi)))


def _cells(case):
    return tuple(max(1, case[k] // case["cell"]) for k in ("nx", "ny", "nz"))


def _views(case, rng):
    # sizes and sample counts belong to the case, cameras and random seeds to the inputs
    sizes = np.random.default_rng(case["views"])
    out = []
    for _ in range(case["views"]):
        frm, at, up, fovy = _orbit(rng.uniform(0, 2 * math.pi), rng.uniform(1.5, 2.3),
                                   rng.uniform(-0.8, 0.8))
        w, h = (int(x) for x in sizes.integers(128, case["width"] + 1, 2))
        out.append({"from": frm, "at": at, "up": up, "fovy": fovy, "width": w, "height": h,
                    "spp": int(sizes.integers(1, case["spp"] + 1)),
                    "seed": int(rng.integers(1, 2**31))})
    return out


def _images(case, rng, n):
    """Network inputs (smooth images seen through noise of every level) and targets."""
    h, w, nc = case["height"], case["width"], case["channels"]
    dev = _device()
    low = torch.from_numpy(rng.random((n, 4 + nc, h // 16 + 2, w // 16 + 2), np.float32)).to(dev)
    base = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear", align_corners=True)
    g = torch.Generator(device=dev)
    g.manual_seed(int(rng.integers(1, 2**31)))
    frames = 2.0 ** rng.integers(0, 13, n)
    x = torch.empty((n, h, w, input_width(nc)), device=dev)
    sd = torch.from_numpy((0.3 / np.sqrt(frames)).astype(np.float32)).to(dev)[:, None, None]
    t = base[:, :3].permute(0, 2, 3, 1)
    noise = torch.randn((n, h, w, 3), device=dev, generator=g)
    x[..., :3] = (t + sd[..., None] * noise).clamp_(min=0)
    x[..., 3] = base[:, 3]
    frac = torch.softmax(4 * torch.cat([torch.zeros_like(base[:, :1]), base[:, 4:]], 1), 1)
    x[..., 4:5 + nc] = frac.permute(0, 2, 3, 1)
    x[..., 5 + nc] = 4.0 * sd * (0.5 + base[:, 0])
    x[..., 6 + nc] = torch.from_numpy((np.log2(frames) / 16).astype(np.float32)).to(dev)[:, None, None]
    return (x.cpu().numpy(), t.contiguous().cpu().numpy(),
            (frames / frames.mean()).astype(np.float32))


def _layers(nc):
    return [(input_width(nc), 32), (32, 32), (32, 64), (64, 64), (64, 96), (96, 96), (160, 64),
            (64, 64), (96, 32), (32, 32), (32, 49)]


def _params(nc, rng):
    """Weights in the order of Denoiser.set_params: [9][cout][cin] and [cout] of each layer;
    the last layer's biases are a Gaussian filter's log weights."""
    out = []
    for i, (cin, cout) in enumerate(_layers(nc)):
        last = i == 10
        out.append(rng.normal(0, 0.02 if last else math.sqrt(2 / (9 * cin)),
                              9 * cout * cin).astype(np.float32))
        y, x = np.mgrid[-3:4, -3:4]
        out.append((-(x * x + y * y) / 4.5).astype(np.float32).ravel() if last else
                   rng.normal(0, 0.02, cout).astype(np.float32))
    return np.concatenate(out)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] in ("infer", "train", "grad"):
        dn = Denoiser(case["width"], case["height"], case["channels"])
        dn.set_params(_params(case["channels"], rng))
        x, t, wt = _images(case, rng, case.get("batch", 1))
        return {"case": case, "dn": dn, "x": x, "t": t, "wt": wt}
    r = MdwtRenderer(0)
    for v in _volumes(case, rng):
        r.push_channel(v)
    r.init(case["mode"], _cells(case), False)
    if case["moments"]:
        r.set_moments(True)
    if case["aov"]:
        r.set_aov(True)
    r.set_frame(case["width"], case["height"], case["spp"], True, (0.0, 0.0, 0.0))
    r.set_camera(*_camera(case, seed))
    if case["gradient"] or case["shadows"]:
        r.set_light((0.3, -1.0, 0.2), case["shadows"], case["gradient"])
    r.set_seed(seed & 0xFFFFFFFF)
    for c, t in enumerate(_tfs(case, rng)):
        r.set_tf(c, t, _opacity(case), (0.0, 1.0))
    if case["kind"] == "batch":
        r.batch_set_launch(case["launch"])
        r.batch_set_views(_views(case, rng))
    return {"case": case, "r": r, "pass": 0, "angle": 0.1 * (seed % 63)}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "infer":
        return state["dn"].infer(state["x"][0])[0]
    if kind == "train":
        loss = state["dn"].train_step(state["x"], state["t"], 1e-3, state["wt"])
        return {"loss": loss, "params": state["dn"].get_params()}
    if kind == "grad":
        g, loss = state["dn"].gradient(state["x"][0], state["t"][0])
        return {"loss": loss, "grad": g}
    r = state["r"]
    if kind == "batch":
        r.batch_reset()
        r.batch_render(case["frames"])
        return [r.batch_read_view(i) for i in range(case["views"])]
    if kind == "view":
        state["pass"] += 1
        if case["edit"]:
            r.set_xf_opacity_scale(state["pass"] % case["channels"],
                                   _opacity(case) * (0.8 + 0.05 * (state["pass"] % 9)))
        else:
            r.set_camera(*_orbit(state["angle"] + 0.02 * state["pass"]))
        r.render(1)
        return r.read_fb()
    r.reset_accumulation()
    r.render(case["frames"])
    if case["moments"]:
        a, m2 = r.read_accum(with_m2=True)
        out = {"image": a, "m2": m2}
    else:
        out = {"image": r.read_accum()}
    if case["aov"]:
        out["aov"] = r.read_aov()
    return out


def work(case):
    """Bytes: every voxel, image, weight and network input read once and every
    output written once. Flops: a tracked ray crosses about one cell per
    macrocell of the grid's longest side and channel (a DDA step and a
    free-flight step, about 40 operations); a marched ray blends every channel
    every half voxel (about 60); the network's multiply-adds, three times over
    with the backward pass."""
    if case["kind"] in ("infer", "train", "grad"):
        n = case["width"] * case["height"]
        px = n * case.get("batch", 1)
        level = [0, 0, 1, 1, 2, 2, 1, 1, 0, 0, 0]
        ls = _layers(case["channels"])
        flops = sum(18 * i * o * (px >> (2 * v)) for (i, o), v in zip(ls, level))
        p = 4 * sum(9 * i * o + o for i, o in ls)
        io = 4 * px * (input_width(case["channels"]) + 3)
        if case["kind"] == "infer":
            return {"bytes": io + p, "flops": flops}
        # weights (and in training both Adam moments) read and written
        return {"bytes": io + (6 if case["kind"] == "train" else 2) * p, "flops": 3 * flops}
    vol = case["channels"] * case["nx"] * case["ny"] * case["nz"] * _BYTES[case["dtype"]]
    px = case["width"] * case["height"]
    if case["kind"] == "batch":
        side = (128 + case["width"]) / 2
        px = case["views"] * side * side * (1 + case["spp"]) / 2
        rays, out = px * case["frames"], 16 * case["views"] * side * side
    else:
        rays = px * case["spp"] * case["frames"]
        out = (4 if case["kind"] == "view" else 16) * px
        if case["moments"]:
            out += 16 * px
        if case["aov"]:
            out += 4 * (2 + case["channels"]) * px
    if case["mode"] >= 6:
        per = 2 * max(case["nx"], case["ny"], case["nz"]) * case["channels"] * 60
    else:
        per = max(_cells(case)) * (case["channels"] if case["mode"] <= 2 else 1) * 40
        if case["gradient"]:
            per += 6 * 60
        if case["shadows"]:
            per *= 2
    return {"bytes": vol + out, "flops": rays * per}


# ------------------------------------------------------- 64-bit references --
def _conv(x, w, b):
    """x [cin][h][w], w [9][cout][cin] -> [cout][h][w], zero padding."""
    c, h, wd = x.shape
    xp = torch.nn.functional.pad(x, (1, 1, 1, 1))
    y = b[:, None]
    for tap in range(9):
        dy, dx = divmod(tap, 3)
        y = y + w[tap] @ xp[:, dy:dy + h, dx:dx + wd].reshape(c, -1)
    return y.reshape(-1, h, wd)


def _network(x, p, nc):
    """x [h][w][inputs] in 64 bits -> the filtered colour [h][w][3]."""
    ls, at = [], 0
    for cin, cout in _layers(nc):
        ls.append((p[at:at + 9 * cout * cin].reshape(9, cout, cin),
                   p[at + 9 * cout * cin:at + 9 * cout * cin + cout]))
        at += 9 * cout * cin + cout
    f = torch.nn.functional

    def cv(i, v):
        return torch.relu(_conv(v, *ls[i]))

    def pool(v):
        return f.avg_pool2d(v[None], 2)[0]

    def up(v):
        return v.repeat_interleave(2, 1).repeat_interleave(2, 2)

    a1 = cv(1, cv(0, x.permute(2, 0, 1)))
    a3 = cv(3, cv(2, pool(a1)))
    a5 = cv(5, cv(4, pool(a3)))
    a7 = cv(7, cv(6, torch.cat([up(a5), a3])))
    z = _conv(cv(9, cv(8, torch.cat([up(a7), a1]))), *ls[10])
    k = torch.softmax(z, 0)
    h, w = x.shape[:2]
    ys, xs = torch.arange(h, device=x.device), torch.arange(w, device=x.device)
    out = 0.0
    for j in range(49):
        sy, sx = (ys + j // 7 - 3).clamp(0, h - 1), (xs + j % 7 - 3).clamp(0, w - 1)
        out = out + k[j][..., None] * x[sy][:, sx][..., :3]
    return out


def _exact_denoiser(case, seed):
    rng = np.random.default_rng(seed)
    nc, dev = case["channels"], _device()
    p = torch.from_numpy(_params(nc, rng)).to(dev, torch.float64)
    xs, ts, wt = _images(case, rng, case.get("batch", 1))
    if case["kind"] == "infer":
        with torch.no_grad():
            return _network(torch.from_numpy(xs[0]).to(dev, torch.float64), p, nc).cpu().numpy()
    p.requires_grad_(True)
    if case["kind"] == "grad":
        wt = np.ones(1)
    loss = 0.0
    for x, t, w in zip(xs, ts, wt):
        y = _network(torch.from_numpy(x).to(dev, torch.float64), p, nc)
        e = ((y - torch.from_numpy(t).to(dev, torch.float64)) ** 2).mean() / len(xs)
        (float(w) * e).backward()
        loss += float(e.detach())
    g = p.grad
    if case["kind"] == "grad":
        return {"loss": loss, "grad": g.cpu().numpy()}
    # the first Adam step: both moments' bias corrections cancel
    return {"loss": loss, "params": (p.detach() - 1e-3 * g / (g.abs() + 1e-8)).cpu().numpy()}


def _philox0(c0, c1, k0, k1):
    """Word 0 of the seven-round Philox4x32 block (c0, c1, 0, 0), int64 tensors."""
    m = 0xFFFFFFFF

    def mul(a, x):  # 32 x 32 -> (hi, lo) in 64-bit integers
        lo, hi = a * (x & 0xFFFF), a * (x >> 16)
        t = lo + ((hi & 0xFFFF) << 16)
        return ((hi >> 16) + (t >> 32)) & m, t & m

    c = [c0, c1, torch.zeros_like(c0), torch.zeros_like(c0)]
    for r in range(7):
        if r:
            k0, k1 = (k0 + 0x9E3779B9) & m, (k1 + 0xBB67AE85) & m
        (h0, l0), (h1, l1) = mul(0xD2511F53, c[0]), mul(0xCD9E8D57, c[2])
        c = [h1 ^ c[1] ^ k0, l1, h0 ^ c[3] ^ k1, l0]
    return c[0]


def _exact_march(case, seed):
    """The ray marchers' image: they are deterministic up to the pixel jitter."""
    rng = np.random.default_rng(seed)
    dev, f64 = _device(), torch.float64
    dims = (case["nx"], case["ny"], case["nz"])
    vols = [torch.from_numpy(v.astype(np.float64)).to(dev) for v in _volumes(case, rng)]
    scale = {"u8": 255.0, "u16": 65535.0}.get(case["dtype"], 1.0)
    tfs = []
    for v, t in zip(vols, _tfs(case, rng)):
        t = t.astype(np.float64)
        t[:, 3] = t[:, 3] ** 3 * float(np.float32(_opacity(case)))
        tfs.append((torch.from_numpy(t).to(dev), min(0.0, float(v.min()) * scale),
                    max(1.0, float(v.max()) * scale)))
    frm, at, up, fovy = _camera(case, seed)
    frm, at, up = (np.array(a, np.float64) for a in (frm, at, up))
    w, h = case["width"], case["height"]
    back = (frm - at) / np.linalg.norm(frm - at)
    u = np.cross(up, back)
    u /= np.linalg.norm(u)
    v = np.cross(back, u)
    hh = math.tan(math.radians(fovy) / 2) * 10.0
    hw = hh * w / h
    llc, hor, ver = (torch.tensor(a, device=dev, dtype=f64)
                     for a in (frm - hw * u - hh * v - 10 * back, 2 * hw * u, 2 * hh * v))
    org = torch.tensor(frm, device=dev, dtype=f64)
    pix = torch.arange(w * h, device=dev)
    px, py = (pix % w).to(f64), (pix // w).to(f64)
    dt = float(np.float32(0.5) * np.float32(1) / np.float32(max(dims)))

    def sample(p, vol):
        idx, fr = [], []
        for k in range(3):
            x = p[:, k] * dims[k] - 0.5
            fl = x.floor()
            fr.append(x - fl)
            i = fl.long()
            idx.append((i.clamp(0, dims[k] - 1), (i + 1).clamp(0, dims[k] - 1)))
        flat, out = vol.reshape(-1), 0.0
        for a in range(8):
            b = (a & 1, a >> 1 & 1, a >> 2)
            wt = 1.0
            for k in range(3):
                wt = wt * (fr[k] if b[k] else 1 - fr[k])
            out = out + wt * flat[(idx[2][b[2]] * dims[1] + idx[1][b[1]]) * dims[0] + idx[0][b[0]]]
        return out * scale

    def lookup(f, tf):
        tab, lo, hi = tf
        x = (f - lo) / (hi - lo) * len(tab) - 0.5
        fl = x.floor()
        a, b = tab[fl.long().clamp(0, len(tab) - 1)], tab[(fl.long() + 1).clamp(0, len(tab) - 1)]
        return a + (x - fl)[:, None] * (b - a)

    def blend(p):
        s = torch.stack([lookup(sample(p, vol), tf) for vol, tf in zip(vols, tfs)])
        al = s[..., 3]
        if case["mode"] == 7:
            best = al.argmax(0)
            o = s.gather(0, best[None, :, None].expand(1, -1, 4))[0]
        elif case["mode"] == 6:
            d = al.sum(0)
            o = (s * al[..., None]).sum(0) / torch.where(d > 0, d, 1.0)[:, None]
        else:
            mo = al.max(0).values
            o = (s * al[..., None]).sum(0) / torch.where(mo > 0, mo, 1.0)[:, None]
            o[:, 3] = mo
        inside = ((p >= 0) & (p <= 1)).all(1) & (al.max(0).values > 0)
        return torch.where(inside[:, None], o, torch.zeros_like(o))

    total = torch.zeros((w * h, 3), device=dev, dtype=f64)
    for frame in range(case["frames"]):
        one = torch.full_like(pix, 1)
        j = (_philox0(one * frame, one * 0, one * (seed & 0xFFFFFFFF), pix) >> 8).to(f64) * 2.0 ** -24
        d = llc + ((px + j) / w)[:, None] * hor + ((py + j) / h)[:, None] * ver - org
        d = d / d.norm(dim=1, keepdim=True)
        a, b = (0.0 - org) / d, (1.0 - org) / d
        t0, t1 = torch.minimum(a, b).amax(1).clamp(min=0), torch.maximum(a, b).amin(1)
        hit = (t1 >= 0) & (t0 < t1)
        rays = hit.nonzero()[:, 0]
        t0, t1, d = t0[rays], t1[rays], d[rays]
        col = torch.zeros((len(rays), 3), device=dev, dtype=f64)
        alpha = torch.zeros(len(rays), device=dev, dtype=f64)
        # the first sample is at the camera, outside the volume; the others trail t by a step
        for i in range(1, int(math.ceil(math.sqrt(3) / dt)) + 2):
            live = (t0 + i * dt < t1) & (alpha < 0.99)
            if not bool(live.any()):
                break
            s = blend(org + d * (t0 + (i - 1) * dt)[:, None])
            k = torch.where(live, (1 - alpha) * s[:, 3], torch.zeros_like(alpha))
            col += s[:, :3] * k[:, None]
            alpha = alpha + k
        # light 1, ambient 0.1, white specular colour at a quarter
        total[rays] += col + 0.1 * (0.75 * col + 0.25)
    img = torch.full((w * h, 4), 1.0 + 1.0 / case["spp"], device=dev, dtype=f64)
    img[:, :3] = total / case["frames"]
    return {"image": img.reshape(h, w, 4).cpu().numpy()}


def exact(case, seed):
    """64-bit references of the denoiser and the ray marchers. The tracking
    modes have none: their images are the outcome of accept / reject decisions
    on 32-bit random numbers."""
    if case["kind"] in ("infer", "train", "grad"):
        return _exact_denoiser(case, seed)
    if case["kind"] == "frames" and case["mode"] >= 6 and case["spp"] == 1:
        return _exact_march(case, seed)
    return None
