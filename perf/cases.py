"""Timed cases of the GI pass: what its users run, at the sizes they run it.

Every case goes through the package's public entry points.  The inputs are
box scenes in the unit-cube room (the project's scene rules) rasterised here
from the seed, four of the visible boxes emissive, so every frame is lit.
`exact` restates the method in 64 bits with plain torch: occupancy, the exact
distance transform and its byte code, the interval march, the bilinear merge,
the gather, and for the learned far field the mip pyramid, the cones and the
network.
"""
import math
import struct

import numpy as np
import torch

import radiancecascade_amd as rc

DEV = "cuda:0"
NEAR, FAR = 0.1, 100.0        # the reference camera's depth planes
THRESHOLD = 1.0               # tile fallback: predicted tile error that takes the plain cascades
CHANNELS = 64                 # network inputs (16 directions x (rgb, transmittance)) and layer width
RADIANCE = 48                 # network outputs that are radiance; output 48 is the error head


# ---- the cases ----------------------------------------------------------------
def _frame(name, w, h, storage="f32", tuned=True, ndc=False, present=False):
    return {"name": name, "kind": "frame", "width": w, "height": h, "storage": storage, "tuned": tuned,
            "ndc": ndc, "present": present, "boxes": 32}


def listed():
    return [
        # the smallest call: a thumbnail or probe view, run once in a while, never tuned
        _frame("frame_256", 256, 256, tuned=False),
        # an interactive renderer's resized window: its own depth buffer (NDC), 16-bit
        # storage, and the presented BGRA8 image
        _frame("present_odd", 1283, 717, storage="bf16", tuned=False, ndc=True, present=True),
        # the headline frame: 1920x1080, 6 levels, fp32, a tuned context
        _frame("frame_1080p", 1920, 1080),
        # the largest single frame: 3840x2160, 7 levels, half storage
        _frame("frame_4k", 3840, 2160, storage="f16"),
        # the learned far field in a real-time loop
        {"name": "learned_1080p", "kind": "learned", "width": 1920, "height": 1080, "storage": "f32", "tuned": True,
         "fallback": False, "boxes": 32},
        # the same with the tile fallback to the plain cascades, odd size, untuned
        {"name": "learned_fallback", "kind": "learned", "width": 1366, "height": 768, "storage": "f16", "tuned": False,
         "fallback": True, "boxes": 32},
        # many cameras at once: one graph launch over views of uneven sizes
        {"name": "batch_16", "kind": "batch", "views": 16, "sizes": 3, "most": 2048, "storage": "f32"},
        # the host boundary of a CPU-side renderer: upload, frame, read back (page-locked)
        {"name": "host_1080p", "kind": "host", "width": 1920, "height": 1080, "boxes": 32},
        # training data: rasterise a scene and write its training rows
        {"name": "rows_1080p", "kind": "rows", "width": 1920, "height": 1080, "boxes": 32},
        # one gradient of the network at the trainer's batch
        {"name": "gradient_16k", "kind": "gradient", "rows": 16384},
        # an epoch of training on rows the caller holds
        {"name": "train_512k", "kind": "train", "rows": 524288, "batch": 16384},
        # the network alone over a feature matrix (validation of a trained network)
        {"name": "network_100k", "kind": "network", "rows": 100003},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi_w, hi_h):
    w = _log_int(rng, lo, hi_w)
    return w, max(lo // 2, min(hi_h, int(w * rng.uniform(0.4, 1.1))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "learned", "batch", "host", "rows", "gradient", "train", "network"])
    if kind == "frame":
        w, h = _size(rng, 64, 3840, 2160)
        c = _frame("", w, h, storage=rng.choice(["f32", "f16", "bf16"]), tuned=rng.random() < 0.5,
                   ndc=rng.random() < 0.5, present=rng.random() < 0.5)
        c["boxes"] = rng.randint(24, 64)
    elif kind == "learned":
        w, h = _size(rng, 256, 1920, 1080)
        c = {"kind": kind, "width": w, "height": h, "storage": rng.choice(["f32", "f16", "bf16"]),
             "tuned": rng.random() < 0.5, "fallback": rng.random() < 0.5, "boxes": rng.randint(24, 64)}
    elif kind == "batch":
        c = {"kind": kind, "views": rng.randint(2, 12), "sizes": rng.randint(0, 1 << 20), "most": _log_int(rng, 512, 2048),
             "storage": rng.choice(["f32", "f16", "bf16"])}
    elif kind in ("host", "rows"):
        w, h = _size(rng, 128, 1920, 1080)
        c = {"kind": kind, "width": w, "height": h, "boxes": rng.randint(24, 64)}
    elif kind == "train":
        batch = rng.choice([4096, 8192, 16384])
        c = {"kind": kind, "rows": max(batch, _log_int(rng, 32768, 524288)), "batch": batch}
    else:
        c = {"kind": kind, "rows": _log_int(rng, 32, 65536 if kind == "gradient" else 131072)}
    c.pop("name", None)
    return c


# ---- inputs -------------------------------------------------------------------
def _boxes(rng, n):
    """[n][12]: lo, hi, albedo, emission; no box reaches into the clear zone around the camera."""
    out = np.zeros((n, 12))
    i = 0
    while i < n:
        c, e = rng.uniform(0, 1, 3), rng.uniform(0.1, 0.4, 3)
        lo, hi = c - e / 2, c + e / 2
        if np.all((lo < 0.65) & (hi > 0.35)):
            continue
        out[i, :3], out[i, 3:6], out[i, 6:9] = lo, hi, rng.uniform(0.2, 0.9, 3)
        i += 1
    return out


def _raster(boxes, w, h):
    """Linear depth [h][w] and the index of the nearest box (-1: the room), in fp64."""
    f = dict(dtype=torch.float64, device=DEV)
    th = 1.0 / math.sqrt(3.0)
    dx = (-((2.0 * (torch.arange(w, **f) + 0.5) / w - 1.0) * th) * (w / h))[None, :].expand(h, w)
    dy = ((1.0 - 2.0 * (torch.arange(h, **f) + 0.5) / h) * th)[:, None].expand(h, w)
    best = torch.full((h, w), 0.5, **f)
    for d in (dx, dy):
        best = torch.minimum(best, 0.5 / d.abs())
    which = torch.full((h, w), -1, dtype=torch.int64, device=DEV)
    for b, box in enumerate(boxes):
        lo, hi = box[:3] - 0.5, box[3:6] - 0.5
        tn = torch.full((h, w), min(lo[2], hi[2]), **f)
        tf = torch.full((h, w), max(lo[2], hi[2]), **f)
        for a, d in ((0, dx), (1, dy)):
            t1, t2 = lo[a] / d, hi[a] / d
            tn, tf = torch.maximum(tn, torch.minimum(t1, t2)), torch.minimum(tf, torch.maximum(t1, t2))
        hit = (tn <= tf) & (tn > 0) & (tn < best)
        best = torch.where(hit, tn, best)
        which = torch.where(hit, b, which)
    return best, which


def _scene(seed, n_boxes, w, h):
    """A lit G-buffer: boxes (four of the visible ones emissive), depth, albedo, emissive."""
    rng = np.random.RandomState(seed % (1 << 32))
    boxes = _boxes(rng, n_boxes)
    depth, which = _raster(boxes, w, h)
    seen = [b for b in torch.unique(which).tolist() if b >= 0]
    for b in rng.permutation(seen)[:4]:
        boxes[b, 9:12] = rng.uniform(1.0, 10.0, 3)
    table = torch.from_numpy(np.concatenate([boxes[:, 6:], [[0.75] * 3 + [0.0] * 3]])).float().to(DEV)
    surface = table[which].permute(2, 0, 1)
    return boxes, depth.float(), surface[:3].contiguous(), surface[3:].contiguous()


def _ndc(depth):
    d = depth.double()
    return (FAR * (d - NEAR) / ((FAR - NEAR) * d)).float()


def _view_sizes(case):
    rng = np.random.RandomState(case["sizes"])
    return [(int(w), int(h)) for w, h in np.exp(rng.uniform(math.log(256), math.log(case["most"]), (case["views"], 2)))]


def _rows(seed, n):
    """Training rows as the cascades give them: features (log(1 + c) rgb, transmittance) of 16 cones, mostly
    dark, and residuals that partly follow them."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    f = dict(device=DEV, generator=g)
    lit = (torch.rand(n, 16, 1, **f) < 0.4).float()
    c = lit * torch.exp(torch.randn(n, 16, 3, **f) - 1.0)
    t = (torch.rand(n, 16, 1, **f) * 1.6 - 0.3).clamp(0.0, 1.0)
    feats = torch.cat([torch.log1p(c), t], -1).reshape(n, CHANNELS)
    noise = torch.randn(n, RADIANCE, **f)
    targets = 0.3 * (c * (1.0 - t)).reshape(n, RADIANCE) - 0.1 + 0.2 * noise * lit.expand(n, 16, 3).reshape(n, RADIANCE)
    return feats.contiguous(), targets.contiguous()


def _with_room(rows):
    """The same rows at the head of a buffer with room for more, as a program that collects rows
    frame by frame keeps them."""
    room = torch.zeros((rows.shape[0] + 64, rows.shape[1]), device=DEV)
    room[:rows.shape[0]] = rows
    return room[:rows.shape[0]]


def _network(seed):
    """He-uniform weights; the output layer's padding columns are zero."""
    rng = np.random.RandomState(seed % (1 << 32))
    layers = []
    for l in range(4):
        w = rng.uniform(-1, 1, (CHANNELS, 64)) * math.sqrt(6.0 / CHANNELS)
        if l == 3:
            w[:, RADIANCE + 1:] = 0.0
        layers += [w.reshape(-1), np.zeros(64)]
    return np.concatenate(layers).astype(np.float32)


def _statistics(feats):
    x = feats.double()
    return x.mean(0).cpu().numpy().astype(np.float32), (1.0 / x.std(0, unbiased=False).clamp(min=1e-3)).cpu().numpy().astype(np.float32)


def _network_inputs(case, seed):
    feats, targets = _rows(seed, case["rows"])
    mean, istd = _statistics(feats) if case["rows"] > 1 else (np.zeros(CHANNELS, np.float32), np.ones(CHANNELS, np.float32))
    return feats, targets / targets.square().mean().sqrt(), _network(seed + 1), mean, istd


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("frame", "learned", "host", "rows"):
        w, h = case["width"], case["height"]
        boxes, depth, albedo, emissive = _scene(seed, case["boxes"], w, h)
        s.update(depth=depth, emissive=emissive, irradiance=torch.empty_like(emissive))
    if kind == "frame":
        if case["ndc"]:
            s["depth"] = _ndc(depth)
        s["stage"] = rc.RadianceCascadeStage(w, h, storage=case["storage"], ndc_depth=(NEAR, FAR) if case["ndc"] else None)
        if case["present"]:
            s.update(albedo=albedo, image=torch.empty((h, w), dtype=torch.int32, device=DEV))
    elif kind == "learned":
        s["stage"] = rc.RadianceCascadeStage(w, h, storage=case["storage"])
        s["stage"].load_weights()
        s["stage"].set_surrogate(True, threshold=THRESHOLD if case["fallback"] else float("inf"))
    elif kind == "host":
        s["stage"] = rc.RadianceCascadeStage(w, h)
        s.update(depth=rc.host_buffer((h, w)), emissive=rc.host_buffer((3, h, w)), irradiance=rc.host_buffer((3, h, w)))
        s["depth"][...] = depth.cpu().numpy()
        s["emissive"][...] = emissive.cpu().numpy()
    elif kind == "rows":
        px, py = rc.probe_grid(w, h, 2)
        s["stage"] = rc.RadianceCascadeStage(w, h)
        s.update(boxes=boxes, depth=torch.empty_like(depth), emissive=torch.empty_like(emissive),
                 feats=torch.empty((px * py, CHANNELS), device=DEV), targets=torch.empty((px * py, RADIANCE), device=DEV))
    elif kind == "batch":
        views = []
        for i, (w, h) in enumerate(_view_sizes(case)):
            _, depth, _, emissive = _scene(seed * 64 + i, 32, w, h)
            views.append((depth, emissive, torch.empty_like(emissive)))
        s.update(views=views, batch=rc.RadianceCascadeBatch(views, storage=case["storage"]))
    elif kind == "train":
        feats, targets = _rows(seed, case["rows"])
        s.update(stage=rc.RadianceCascadeStage(64, 64), feats=feats, targets=targets, scaled=_with_room(targets))
    else:
        feats, targets, params, mean, istd = _network_inputs(case, seed)
        s.update(stage=rc.RadianceCascadeStage(64, 64), feats=feats, targets=_with_room(targets),
                 z=torch.empty((case["rows"], 64), device=DEV),
                 grad=torch.empty(params.size, device=DEV), loss=torch.empty(1, device=DEV))
        s["stage"].mlp_set(params, mean, istd, 1.0)
    if case.get("tuned"):
        s["stage"].autotune(s["depth"], s["emissive"], s["irradiance"], iters=3)
    return s


# ---- one pass -----------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("frame", "learned"):
        s["stage"].run_device(s["depth"], s["emissive"], s["irradiance"])
        if not case.get("present"):
            return s["irradiance"]
        s["stage"].composite(s["albedo"], s["emissive"], s["irradiance"], s["image"])
        return {"irradiance": s["irradiance"], "image": s["image"]}
    if kind == "host":
        s["stage"].update(s["depth"], s["emissive"])
        return s["stage"].render(s["irradiance"])
    if kind == "batch":
        s["batch"].run()
        return [v[2] for v in s["views"]]
    if kind == "rows":
        rc.gbuffer_raster(s["boxes"], case["width"], case["height"], s["depth"], None, s["emissive"])
        s["stage"].surrogate_samples(s["depth"], s["emissive"], s["feats"], s["targets"])
        return {"depth": s["depth"], "emissive": s["emissive"], "feats": s["feats"], "targets": s["targets"]}
    if kind == "gradient":
        s["stage"].mlp_gradient(s["feats"], s["targets"], s["grad"], s["loss"])
        return {"grad": s["grad"], "loss": s["loss"]}
    if kind == "network":
        s["stage"].mlp_forward(s["feats"], s["z"])
        return s["z"]
    # training scales its targets in place: a program that trains again passes a copy
    s["scaled"].copy_(s["targets"])
    report = s["stage"].train_surrogate_rows(s["feats"], s["scaled"], epochs=1, batch=case["batch"], seed=1)
    return {"loss": report["epoch_loss"], **s["stage"].mlp_get()}


# ---- what a pass cannot do without ---------------------------------------------
def _frame_work(w, h, levels=None, present=False):
    """Each input read and each output written once; per ray one sample of the field (two multiply-adds and a
    comparison per axis) and one bilinear merge of three channels."""
    levels = levels or rc.levels_for_coverage(w, h)
    rays = sum(rc.level_rays(w, h, i) for i in range(levels))
    return w * h * (16 + 12 + (16 if present else 0)), rays * (8 + 21)


def work(case):
    kind = case["kind"]
    n = case.get("rows", 0)
    params = 4 * (CHANNELS * 64 + 64)
    if kind in ("frame", "host"):
        b, f = _frame_work(case["width"], case["height"], present=case.get("present", False))
    elif kind == "learned":
        b, f = _frame_work(case["width"], case["height"], levels=2)
        px, py = rc.probe_grid(case["width"], case["height"], 2)
        f += 2 * 4 * CHANNELS * 64 * px * py
    elif kind == "batch":
        each = [_frame_work(w, h) for w, h in _view_sizes(case)]
        b, f = sum(x for x, _ in each), sum(x for _, x in each)
    elif kind == "rows":
        px, py = rc.probe_grid(case["width"], case["height"], 2)
        f = _frame_work(case["width"], case["height"])[1] + 8 * case["boxes"] * case["width"] * case["height"]
        b = 16 * case["width"] * case["height"] + px * py * 4 * (CHANNELS + RADIANCE)
    elif kind == "network":
        b, f = n * 4 * (CHANNELS + 64) + 4 * params, n * 2 * 4 * CHANNELS * 64
    elif kind == "gradient":
        b, f = n * 4 * (CHANNELS + RADIANCE) + 8 * params, n * 2 * (3 * 4 - 1) * CHANNELS * 64
    else:
        # the rows once for their statistics and once for the epoch
        b, f = 2 * n * 4 * (CHANNELS + RADIANCE), n * 2 * (3 * 4 - 1) * CHANNELS * 64
    return {"bytes": b, "flops": f}


# ---- the same in 64 bits ---------------------------------------------------------
def _occupied(depth, emissive):
    d, e = depth.double(), emissive
    occ = (e > 0).any(0)
    for a in (0, 1):
        step = d.diff(dim=a)
        edge = torch.zeros_like(occ)
        n = step.shape[a]
        edge.narrow(a, 0, n).logical_or_(step > 0.05 * d.narrow(a, 0, n))
        edge.narrow(a, 1, n).logical_or_(-step > 0.05 * d.narrow(a, 1, n))
        occ = occ | edge
    return occ


def _field(occ):
    """The byte code's value of the distance to the nearest occupied pixel."""
    h, w = occ.shape
    y = torch.arange(h, device=DEV, dtype=torch.int32)[:, None]
    up = torch.where(occ, y, -20000).cummax(0).values
    down = torch.where(occ, y, 20000 + h).flip(0).cummin(0).values.flip(0)
    g2 = torch.minimum(y - up, down - y).clamp(max=20000).square()
    x = torch.arange(w, device=DEV, dtype=torch.int32)
    dx2 = (x[:, None] - x[None, :]).square()
    d2 = torch.empty_like(g2)
    rows = max(1, (1 << 28) // (w * w))
    for r in range(0, h, rows):
        d2[r:r + rows] = (dx2[None] + g2[r:r + rows, None, :]).amin(-1)
    d = d2.double().sqrt().floor()
    return torch.where(d < 128, d, torch.where(d < 2160, 128 + 16 * ((d - 128) / 16).floor(), 2160.0))


def _grid(w, h, level):
    s = 2 << level
    return -(-w // s), -(-h // s)


def _march(field, emissive, level):
    """rgb [PY][PX][N][3] of every ray of a level and whether it went on ([PY][PX][N])."""
    h, w = field.shape
    px, py = _grid(w, h, level)
    n, s = 4 << (2 * level), 2 << level
    t0, t1 = 2 * (4 ** level - 1) / 3, 2 * (4 ** (level + 1) - 1) / 3
    th = 2.0 * math.pi * (torch.arange(n, device=DEV, dtype=torch.float64) + 0.5) / n
    shape = (py, px, n)
    dx, dy = th.cos().expand(shape).reshape(-1), th.sin().expand(shape).reshape(-1)
    cx = ((torch.arange(px, device=DEV).double() + 0.5) * s)[None, :, None].expand(shape).reshape(-1)
    cy = ((torch.arange(py, device=DEV).double() + 0.5) * s)[:, None, None].expand(shape).reshape(-1)
    t = torch.full_like(cx, t0)
    ray = torch.arange(cx.numel(), device=DEV)
    hit = torch.full((cx.numel(),), -1, dtype=torch.int64, device=DEV)
    flat = field.reshape(-1)
    while ray.numel():
        x, y = (cx + t * dx).floor().long(), (cy + t * dy).floor().long()
        ok = (x >= 0) & (x < w) & (y >= 0) & (y < h)
        q = torch.where(ok, y * w + x, 0)
        d = flat[q]
        found = ok & (d < 0.5)
        hit[ray[found]] = q[found]
        t = t + d.clamp(min=1.0)
        on = ok & ~found & (t < t1)
        ray, t, cx, cy, dx, dy = (v[on] for v in (ray, t, cx, cy, dx, dy))
    rgb = emissive.double().reshape(3, -1).T[hit.clamp(min=0)] * (hit >= 0).double()[:, None]
    return rgb.reshape(py, px, n, 3), (hit < 0).reshape(shape)


def _bilinear(upper, px, py):
    """The upper grid's texels [UY][UX][...] at the grid of half its spacing."""
    def axis(n, un):
        p = torch.arange(n, device=DEV)
        base = (p - 1) >> 1
        w1 = torch.where(p % 2 == 1, 0.25, 0.75).double()
        return base.clamp(0, un - 1), (base + 1).clamp(0, un - 1), w1
    x0, x1, wx = axis(px, upper.shape[1])
    y0, y1, wy = axis(py, upper.shape[0])
    more = [1] * (upper.dim() - 2)
    rows = upper[:, x0] * (1 - wx).reshape(1, -1, *more) + upper[:, x1] * wx.reshape(1, -1, *more)
    return rows[y0] * (1 - wy).reshape(-1, 1, *more) + rows[y1] * wy.reshape(-1, 1, *more)


def _merge(field, emissive, level, upper):
    rgb, on = _march(field, emissive, level)
    if upper is not None:
        rgb = rgb + on[..., None] * _bilinear(upper, rgb.shape[1], rgb.shape[0])
    py, px, n, _ = rgb.shape
    return rgb.reshape(py, px, n // 4, 4, 3).mean(3)


def _gather(a0, w, h):
    return _bilinear(a0[:, :, 0], w, h).permute(2, 0, 1).contiguous()


def _irradiance(depth, emissive, down_to=0):
    """The plain frame; or its merged level `down_to`."""
    h, w = depth.shape
    field = _field(_occupied(depth, emissive))
    levels, a = rc.levels_for_coverage(w, h), None
    for i in range(levels - 1, down_to - 1, -1):
        a = _merge(field, emissive, i, a)
    return a if down_to else _gather(a, w, h)


def _pyramid(occ, emissive):
    """Cells [h][w][8] per mip level, one cell of zeros around: mean emission, emitter area, the fractions of
    pixel columns and rows with an emitter, then with a dark occluder."""
    em = (emissive > 0).any(0)
    dark = occ & ~em
    f = torch.cat([emissive.double() * em, torch.stack([em, em, em, dark, dark]).double()])
    top = 1
    while (1 << top) < max(occ.shape):
        top += 1
    levels = [None]
    for _ in range(top):
        f = torch.nn.functional.pad(f, (0, f.shape[2] % 2, 0, f.shape[1] % 2))
        tl, tr, bl, br = f[:, ::2, ::2], f[:, ::2, 1::2], f[:, 1::2, ::2], f[:, 1::2, 1::2]
        mean = (tl + tr + bl + br)[:4] / 4
        x = (torch.maximum(tl, bl) + torch.maximum(tr, br)) / 2
        y = (torch.maximum(tl, tr) + torch.maximum(bl, br)) / 2
        f = torch.cat([mean, x[4:5], y[5:6], x[6:7], y[7:8]])
        levels.append(torch.nn.functional.pad(f, (1, 1, 1, 1)).permute(1, 2, 0).contiguous())
    return levels


def _trace(levels, w, h, grid_level, steps):
    px, py = _grid(w, h, grid_level)
    s = 2 << grid_level
    th = 2.0 * math.pi * (torch.arange(16, device=DEV).double() + 0.5) / 16
    dx, dy = th.cos()[None, None], th.sin()[None, None]
    cx = ((torch.arange(px, device=DEV).double() + 0.5) * s)[None, :, None]
    cy = ((torch.arange(py, device=DEV).double() + 0.5) * s)[:, None, None]
    through = torch.ones((py, px, 16), dtype=torch.float64, device=DEV)
    light = torch.zeros((py, px, 16, 3), dtype=torch.float64, device=DEV)
    live = torch.ones((py, px, 16), dtype=torch.bool, device=DEV)
    for t, m, re in steps:
        cells = levels[m]
        ch, cw = cells.shape[0] - 2, cells.shape[1] - 2
        fx, fy = (t * dx + cx) / (1 << m) - 0.5, (t * dy + cy) / (1 << m) - 0.5
        x0, y0 = fx.floor().long(), fy.floor().long()
        ax, ay = (fx - x0)[..., None], (fy - y0)[..., None]
        live = live & (x0 >= -1) & (x0 < cw) & (y0 >= -1) & (y0 < ch)
        xs, ys = (x0 + 1).clamp(0, cw), (y0 + 1).clamp(0, ch)
        v = ((cells[ys, xs] * (1 - ax) + cells[ys, xs + 1] * ax) * (1 - ay) +
             (cells[ys + 1, xs] * (1 - ax) + cells[ys + 1, xs + 1] * ax) * ay)
        ce, co = (dy * dy * v[..., i] + dx * dx * v[..., i + 1] for i in (4, 6))
        ae = 1 - (1 - ce.clamp(max=0.999)) ** re
        ao = 1 - (1 - co.clamp(max=0.999)) ** (3 * re)
        radiance = torch.where(v[..., 3:4] > 0, v[..., :3] / v[..., 3:4].clamp(min=1e-300), 0.0)
        light = light + (live * through * ae)[..., None] * radiance
        through = torch.where(live, through * (1 - (ae + ao).clamp(max=1.0)), through)
        live = live & (through >= 1e-4)
    return light, through


def _cones(occ, emissive):
    """The level-2 probes' 16 cones: radiance [QY][QX][16][3] and transmittance."""
    h, w = occ.shape
    levels = _pyramid(occ, emissive)
    near, far, t = [], [], 10.0
    while t < math.hypot(w, h) + 2.0 and len(near) + len(far) < 64:
        dia = max(2.0 * t * math.tan(math.pi / 16), 1.0)
        m = min(max(int(math.floor(math.log2(dia))), 1), len(levels) - 1)
        (near if t < 60.0 else far).append((t, m, min(0.75 * dia, float(1 << m)) / (1 << m)))
        t += 0.75 * dia
    light, through = _trace(levels, w, h, 2, near)
    light3, through3 = _trace(levels, w, h, 3, far)
    py, px = through.shape[:2]
    return light + through[..., None] * _bilinear(light3, px, py), through * _bilinear(through3, px, py)


def _features(light, through):
    return torch.cat([torch.log1p(light), through[..., None]], -1).reshape(-1, CHANNELS)


def _layers(params):
    p = torch.from_numpy(np.asarray(params, np.float64)).to(DEV)
    step = CHANNELS * 64 + 64
    return [(p[i:i + CHANNELS * 64].reshape(CHANNELS, 64), p[i + CHANNELS * 64:i + step]) for i in range(0, 4 * step, step)]


def _forward(layers, feats, mean, istd):
    a = (feats.double() - torch.as_tensor(mean, device=DEV).double()) * torch.as_tensor(istd, device=DEV).double()
    for l, (w, b) in enumerate(layers):
        a = a @ w + b
        a = a.relu() if l < 3 else a
    return a


def _loss(z, targets):
    """Mean squared residual plus the error head's fit to the log of each row's own error."""
    square = (z[:, :RADIANCE] - targets.double()).square()
    wanted = (square.detach().mean(1) + 1e-2).log()
    return square.mean() + 0.05 * (z[:, RADIANCE] - wanted).square().mean()


def _packaged():
    with open(rc.packaged_weights(), "rb") as f:
        blob = f.read()
    v = np.frombuffer(blob, np.float32, offset=32)
    return v[2 * CHANNELS:], v[:CHANNELS], v[CHANNELS:2 * CHANNELS], struct.unpack_from("<f", blob, 24)[0]


def _learned(depth, emissive, fallback):
    h, w = depth.shape
    occ = _occupied(depth, emissive)
    field = _field(occ)
    params, mean, istd, scale = _packaged()
    light, through = _cones(occ, emissive)
    qy, qx = through.shape[:2]
    z = _forward(_layers(params), _features(light, through), mean, istd).reshape(qy, qx, 64)
    a2 = (light + scale * z[..., :RADIANCE].reshape(qy, qx, 16, 3)).clamp(min=0.0)
    a1 = _merge(field, emissive, 1, a2)
    if fallback:
        py, px = a1.shape[:2]
        ty, tx = -(-qy // 8), -(-qx // 8)
        err = torch.full((ty * 8, tx * 8), math.nan, dtype=torch.float64, device=DEV)
        err[:qy, :qx] = z[..., RADIANCE].exp()
        flagged = err.reshape(ty, 8, tx, 8).nanmean((1, 3)) > THRESHOLD
        mask = flagged.repeat_interleave(16, 0).repeat_interleave(16, 1)[:py, :px]
        a1 = torch.where(mask[..., None, None], _irradiance(depth, emissive, 1), a1)
    return _gather(_merge(field, emissive, 0, a1), w, h)


def _mix64(states):
    z = states
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _stream(seed, n):
    """n outputs of SplitMix64."""
    with np.errstate(over="ignore"):
        return _mix64(np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, n + 1, dtype=np.uint64))


def _trained(feats, targets, batch, seed=1, lr=2e-3):
    n = feats.shape[0]
    x = feats.double()
    mean = x.mean(0)
    istd = 1.0 / x.std(0, unbiased=False).clamp(min=1e-3)
    scale = targets.double().square().mean().sqrt()
    u = (_stream(seed, 4 * CHANNELS * 64) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53
    w = ((2.0 * u - 1.0) * math.sqrt(6.0 / CHANNELS)).reshape(4, CHANNELS, 64)
    w[3, :, :RADIANCE] *= 0.5
    w[3, :, RADIANCE + 1:] = 0.0
    p = [torch.from_numpy(v.copy()).to(DEV).requires_grad_() for l in w for v in (l, np.zeros(64))]
    order = list(range(n))
    draws = _stream(seed ^ 0x5DEECE66D, n - 1)
    for i, j in zip(range(n - 1, 0, -1), (draws % np.arange(n, 1, -1, dtype=np.uint64)).tolist()):
        order[i], order[j] = order[j], order[i]
    order = torch.tensor(order, device=DEV)
    m, v, total = [torch.zeros_like(q) for q in p], [torch.zeros_like(q) for q in p], 0.0
    steps = n // batch
    for k in range(steps):
        at = order[k * batch:(k + 1) * batch]
        loss = _loss(_forward(list(zip(p[::2], p[1::2])), feats[at], mean, istd), targets[at].double() / scale)
        grads = torch.autograd.grad(loss, p)
        total += float(loss.detach())
        with torch.no_grad():
            for q, g, mq, vq in zip(p, grads, m, v):
                mq.mul_(0.9).add_(g, alpha=0.1)
                vq.mul_(0.999).add_(g * g, alpha=0.001)
                q.sub_(lr * (mq / (1 - 0.9 ** (k + 1))) / ((vq / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8))
    flat = torch.cat([q.detach().reshape(-1) for q in p])
    return {"loss": [total / steps], "params": flat, "in_mean": mean, "in_istd": istd, "out_scale": float(scale)}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("frame", "host", "learned", "rows"):
        _, depth, _, emissive = _scene(seed, case["boxes"], case["width"], case["height"])
    if kind in ("frame", "host"):
        if case.get("ndc"):
            depth = NEAR * FAR / (FAR - _ndc(depth).double() * (FAR - NEAR))
        irradiance = _irradiance(depth, emissive)
        # the image is bytes: whole values, equal or not
        return {"irradiance": irradiance, "image": None} if case.get("present") else irradiance
    if kind == "learned":
        return _learned(depth, emissive, case["fallback"])
    if kind == "batch":
        scenes = [_scene(seed * 64 + i, 32, w, h) for i, (w, h) in enumerate(_view_sizes(case))]
        return [_irradiance(depth, emissive) for _, depth, _, emissive in scenes]
    if kind == "rows":
        light, through = _cones(_occupied(depth, emissive), emissive)
        level2 = _irradiance(depth, emissive, 2)
        return {"depth": depth.double(), "emissive": emissive.double(), "feats": _features(light, through),
                "targets": (level2 - light).reshape(-1, RADIANCE)}
    if kind == "train":
        return _trained(*_rows(seed, case["rows"]), case["batch"])
    feats, targets, params, mean, istd = _network_inputs(case, seed)
    layers = _layers(params)
    if kind == "network":
        return _forward(layers, feats, mean, istd)
    flat = [p.requires_grad_() for layer in layers for p in layer]
    loss = _loss(_forward(layers, feats, mean, istd), targets)
    grad = torch.cat([g.reshape(-1) for g in torch.autograd.grad(loss, flat)])
    return {"grad": grad, "loss": loss.detach().reshape(1)}
