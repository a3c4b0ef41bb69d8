"""The work that users of this framework have it do, as a list of timed cases.

Each case is one call (or one training step) through a public entry point, on
inputs of the kind the call meets in use: a textured scene of slanted planes,
its right view warped by the true disparity with sensor noise and filled
occlusions.  `listed()` gives the fixed cases, `draw()` more of the same
ranges; `exact()` restates the algorithms in plain torch (integers and
float64).
"""
from __future__ import annotations

import random

import numpy as np
import torch

from fasterstereocuda_amd.batch import SgmBatch
from fasterstereocuda_amd.diff_sgm import diff_sgm
from fasterstereocuda_amd.pyramid import FasterStereoCuda, SgmPyramid, StereoOption1
from fasterstereocuda_amd.stereo import CuSGMOption, StereoCuda

INVALID = -999999.0
FORMATS = ((450, 375), (640, 480), (1242, 375), (1280, 720), (1920, 1080))
TEMPERATURE = 0.1


# ------------------------------------------------------------------ cases
def _pair(name, w, h, d, *, host=False, cs=1, p1=10, p2=150, min_d=0, right=False):
    return {"name": name, "kind": "pair_host" if host else "pair", "w": w, "h": h, "d": d,
            "cs": cs, "p1": p1, "p2": p2, "min_d": min_d, "right": right}


def listed():
    return [
        # a thumbnail or a tracked patch, device-resident: launches and the
        # latency of 160 steps are all there is
        _pair("pair_160x120_d64", 160, 120, 64),
        # the reference console's call: host images in, host map out, at its
        # own sample's size with its default 5x5 census and penalties
        _pair("host_450x375_d64_5x5", 450, 375, 64, host=True, cs=0, p1=8, p2=32),
        # one driving frame as it arrives from a camera, both maps wanted
        _pair("pair_1242x375_d64", 1242, 375, 64, right=True),
        # an HD frame with a wider search, one pair at a time
        _pair("pair_1920x1080_d128", 1920, 1080, 128),
        # an odd-sized crop with the 5x5 census, a 256 range and an offset
        _pair("pair_1117x573_d256_5x5", 1117, 573, 256, cs=0, p1=8, p2=32, min_d=-16),
        # a large aerial or survey image searched densely in one level
        _pair("pair_4800x3409_d256", 4800, 3409, 256),
        # offline processing of a driving sequence, 32 frames per call
        {"name": "batch_32x1242x375_d64", "kind": "batch", "n": 32, "w": 1242, "h": 375, "d": 64},
        # a mixed queue: pairs of five formats and two ranges in one call
        {"name": "batch_uneven_24", "kind": "uneven", "n": 24, "mix": 3},
        # the large image by the pyramid, window 16, device-resident
        {"name": "pyramid_4800x3409_w16", "kind": "pyramid", "w": 4800, "h": 3409, "max_disp": 256,
         "layers": 3, "window": 16},
        # the FasterStereoCuda class on host images with its own schedule
        # (5x5, window 32, LR check, peak removal)
        {"name": "faster_1281x719_l2", "kind": "faster", "w": 1281, "h": 719, "max_disp": 128,
         "layers": 2},
        # training on small crops: forward and backward of the FP32 form
        {"name": "diff_2x119x321_d64", "kind": "diff", "n": 2, "h": 119, "w": 321, "d": 64},
        # training on full driving frames, batch 8
        {"name": "diff_8x375x1242_d128", "kind": "diff", "n": 8, "h": 375, "w": 1242, "d": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["pair", "pair", "pair", "large", "pair_host", "batch", "uneven", "pyramid",
                       "faster", "diff", "diff"])
    if kind in ("pair", "pair_host"):
        d = rng.choice([64, 64, 128, 256])
        w = _log_int(rng, 96, 1920 if kind == "pair" else 1300)
        h = _log_int(rng, 64, 1080 if kind == "pair" else 720)
        while w * h * d > 1920 * 1080 * 128:
            h = max(64, h // 2)
        cs = rng.choice([0, 1, 1])
        p1, p2 = (10, 150) if cs else (8, 32)
        return {"kind": kind, "w": w, "h": h, "d": d, "cs": cs, "p1": p1, "p2": p2,
                "min_d": rng.choice([0, 0, 0, -16, 7]), "right": rng.random() < 0.3}
    if kind == "large":
        w, h = _log_int(rng, 1920, 4800), _log_int(rng, 1080, 3409)
        return {"kind": "pair", "w": w, "h": h, "d": rng.choice([128, 256]), "cs": 1, "p1": 10,
                "p2": 150, "min_d": 0, "right": False}
    if kind == "batch":
        d = rng.choice([64, 64, 128])
        w, h = _log_int(rng, 320, 1920), _log_int(rng, 240, 1080)
        most = max(1, 32 * 1242 * 375 * 64 // (w * h * d))
        return {"kind": "batch", "n": min(48, _log_int(rng, 1, most)) if most > 1 else 1,
                "w": w, "h": h, "d": d}
    if kind == "uneven":
        return {"kind": "uneven", "n": rng.randint(6, 24), "mix": rng.randint(4, 10 ** 6)}
    if kind == "pyramid":
        return {"kind": "pyramid", "w": _log_int(rng, 640, 4800), "h": _log_int(rng, 480, 3409),
                "max_disp": rng.choice([128, 256]), "layers": rng.choice([2, 3, 3]),
                "window": rng.choice([16, 16, 32])}
    if kind == "faster":
        return {"kind": "faster", "w": _log_int(rng, 320, 1920), "h": _log_int(rng, 240, 1080),
                "max_disp": rng.choice([64, 128]), "layers": rng.choice([1, 2, 3])}
    d = rng.choice([64, 128, 128, 256])
    w, h = _log_int(rng, 64, 1242), _log_int(rng, 48, 375)
    most = max(1, 8 * 375 * 1242 * 128 // (w * h * d))
    return {"kind": "diff", "n": min(_log_int(rng, 1, 8), most), "h": h, "w": w, "d": d}


# ----------------------------------------------------------------- inputs
def _scene(seed, h, w, d, min_d=0):
    """A rectified pair on the GPU: (left, right) uint8 [h, w]."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)

    def rand(*shape):
        return torch.rand(*shape, generator=g, device=dev)

    tex = torch.zeros(h, w, device=dev)
    amp = 1.0
    for cell in (16, 8, 4, 2):
        grid = rand(1, 1, h // cell + 2, w // cell + 2)
        tex += amp * torch.nn.functional.interpolate(grid, size=(h, w), mode="bilinear",
                                                     align_corners=True)[0, 0]
        amp *= 0.5
    left = ((tex - tex.min()) * (255.0 / (tex.max() - tex.min()))).round()
    # slanted planes on a Voronoi partition
    lo, hi = float(max(min_d, 0) + 2), float(min(min_d + d - 4, w // 2))
    hi = max(hi, lo + 1.0)
    n = 6 if h * w < 1 << 20 else 24
    c = rand(n, 5).double().cpu().numpy()
    ys = torch.arange(h, device=dev, dtype=torch.float32)[:, None]
    xs = torch.arange(w, device=dev, dtype=torch.float32)[None, :]
    best = torch.full((h, w), float("inf"), device=dev)
    disp = torch.zeros(h, w, device=dev)
    for cy, cx, base, sx, sy in c:
        dy, dx = ys - float(cy * h), xs - float(cx * w)
        dist = dy * dy + dx * dx
        plane = lo + float(base) * (hi - lo) + float(0.08 * sx - 0.04) * dx + float(0.08 * sy - 0.04) * dy
        near = dist < best
        best = torch.where(near, dist, best)
        disp = torch.where(near, plane, disp)
    disp = disp.clamp(lo, hi)
    # forward warp; the larger disparity wins a column
    xr = (xs - disp).round().long()
    ok = (xr >= 0) & (xr < w)
    key = ((disp * 64).long() << 8) | left.long()
    tgt = (torch.arange(h, device=dev)[:, None] * w + xr)[ok]
    hit = torch.full((h * w,), -1, dtype=torch.long, device=dev)
    hit.scatter_reduce_(0, tgt, key[ok], "amax")
    right = torch.where(hit.view(h, w) >= 0, (hit.view(h, w) & 255).float(), rand(h, w) * 255.0)
    right = right + 2.0 * torch.randn(h, w, generator=g, device=dev)
    return left.to(torch.uint8), right.round().clamp(0, 255).to(torch.uint8)


def _mix(case):
    """(w, h, d) of the pairs of an uneven batch."""
    r = random.Random(case["mix"])
    return [r.choice(FORMATS) + (r.choice([64, 128]),) for _ in range(case["n"])]


def _images(case, seed):
    """The (left, right) device images of a case, one entry per pair."""
    k = case["kind"]
    if k in ("pair", "pair_host"):
        shapes = [(case["w"], case["h"], case["d"])]
    elif k == "batch":
        shapes = [(case["w"], case["h"], case["d"])] * case["n"]
    elif k == "uneven":
        shapes = _mix(case)
    elif k == "diff":
        shapes = [(case["w"], case["h"], case["d"])] * case["n"]
    else:
        shapes = [(case["w"], case["h"], case["max_disp"])]
    return [_scene(seed * 1000 + i, h, w, d, case.get("min_d", 0))
            for i, (w, h, d) in enumerate(shapes)]


def _diff_inputs(case, seed):
    """Normalised Hamming costs of the pairs, per-pixel penalties and the
    gradient that arrives from the loss."""
    n, h, w, d = case["n"], case["h"], case["w"], case["d"]
    cost = torch.empty(n, h, w, d, device="cuda")
    for b, (left, right) in enumerate(_images(case, seed)):
        cl, cr = _census(left[None], 1, False), _census(right[None], 1, True)
        cost[b] = _cost(cl, cr, 0, d, True, 1)[0].float() / 63.0
    g = torch.Generator(device="cuda").manual_seed(seed * 1000 + 777)
    p1 = torch.rand(n, h, w, generator=g, device="cuda") * 0.15 + 0.05
    p2 = torch.rand(n, h, w, generator=g, device="cuda") * 1.5 + 0.5
    up = torch.randn(n, h, w, generator=g, device="cuda") / (n * h * w)
    return cost, p1, p2, up


def _option(case):
    return CuSGMOption.benchmark(cs_type=case.get("cs", 1), p1=case.get("p1", 10),
                                 p2_init=case.get("p2", 150))


def prepare(case, seed):
    k = case["kind"]
    if k == "diff":
        cost, p1, p2, up = _diff_inputs(case, seed)
        return {"kind": k, "in": [t.requires_grad_(True) for t in (cost, p1, p2)], "up": up}
    images = _images(case, seed)
    left, right = images[0]
    if k in ("pair", "pair_host"):
        st = StereoCuda()
        if not st.Init(case["w"], case["h"], case["min_d"], case["d"], _option(case)):
            raise RuntimeError(st.last_error)
        if k == "pair":
            out = [torch.empty(case["h"], case["w"], device="cuda") for _ in range(1 + case["right"])]
            return {"kind": k, "st": st, "in": (left, right), "out": out}
        out = [np.empty((case["h"], case["w"]), np.float32) for _ in range(1 + case["right"])]
        return {"kind": k, "st": st, "in": (left.cpu().numpy(), right.cpu().numpy()), "out": out}
    if k in ("batch", "uneven"):
        ds = [s[2] for s in _mix(case)] if k == "uneven" else [case["d"]] * case["n"]
        pairs = [{"left": a, "right": b, "disp_left": torch.empty(a.shape, device="cuda"),
                  "min_disparity": 0, "disp_range": d} for (a, b), d in zip(images, ds)]
        return {"kind": k, "batch": SgmBatch(pairs, _option(case)),
                "out": [p["disp_left"] for p in pairs]}
    if k == "pyramid":
        pyr = SgmPyramid(case["w"], case["h"], 0, case["max_disp"], case["layers"], case["window"],
                         _option(case))
        return {"kind": k, "pyr": pyr, "in": (left, right),
                "out": torch.empty(case["h"], case["w"], device="cuda")}
    fs = FasterStereoCuda()
    if not fs.Init(StereoOption1(case["w"], case["h"], 0, case["max_disp"], case["layers"])):
        raise RuntimeError(fs.last_error)
    return {"kind": k, "fs": fs, "in": (left.cpu().numpy(), right.cpu().numpy()),
            "out": np.empty((case["h"], case["w"]), np.float32)}


def run(state):
    k = state["kind"]
    if k == "diff":
        disp = diff_sgm(*state["in"], TEMPERATURE)
        return (disp.detach(), *torch.autograd.grad(disp, state["in"], state["up"]))
    if k == "pair":
        ok = state["st"].match_device(*state["in"], *state["out"])
    elif k == "pair_host":
        ok = state["st"].Match(*state["in"], *state["out"])
    elif k in ("batch", "uneven"):
        state["batch"].run()
        ok = True
    elif k == "pyramid":
        state["pyr"].match_device(*state["in"], state["out"])
        ok = True
    else:
        ok = state["fs"].Match(*state["in"], state["out"])
    if not ok:
        raise RuntimeError("match failed")
    return state["out"]


def work(case):
    """Images in, maps out; the integer operations of the recurrence: a cost
    (4) and, per direction, three additions, three minima and the running
    minimum (8) per cell and view, then the sum and minimum of the four."""
    k = case["kind"]
    if k == "diff":
        cells = case["n"] * case["h"] * case["w"] * case["d"]
        pix = case["n"] * case["h"] * case["w"]
        # cost in, its gradient out; penalties and their gradients, up, map
        return {"bytes": 8 * cells + 24 * pix, "flops": 4 * 20 * cells}
    per_cell = 4 + 4 * 8 + 5
    if k in ("pair", "pair_host"):
        pix = case["w"] * case["h"]
        return {"bytes": pix * (2 + 4 + 4 * case["right"]), "flops": 2 * per_cell * pix * case["d"]}
    if k == "batch":
        pix = case["n"] * case["w"] * case["h"]
        return {"bytes": pix * 6, "flops": 2 * per_cell * pix * case["d"]}
    if k == "uneven":
        mix = _mix(case)
        return {"bytes": sum(w * h * 6 for w, h, _ in mix),
                "flops": sum(2 * per_cell * w * h * d for w, h, d in mix)}
    window = case["window"] if k == "pyramid" else FasterStereoCuda.LEVEL_RANGE
    top = case["layers"] - 1
    cells = sum((case["w"] >> i) * (case["h"] >> i) * window for i in range(top))
    rng = _interval(case)
    cells += 2 * (case["w"] >> top) * (case["h"] >> top) * rng
    return {"bytes": case["w"] * case["h"] * 6, "flops": per_cell * cells}


# ------------------------------------------------ the same results, plainly
def _census(img, cs, is_right):
    """Census words [n, h, w] int64 of images [n, h, w]; bits of darker
    neighbours in raster order, border pixels constant."""
    rw, rh = (4, 3) if cs else (2, 2)
    n, h, w = img.shape
    out = torch.full((n, h, w), 0xFFFFFFFF if is_right else 0, dtype=torch.long, device=img.device)
    if h <= 2 * rh or w <= 2 * rw:
        return out
    c = img[:, rh:h - rh, rw:w - rw]
    v = torch.zeros(c.shape, dtype=torch.long, device=img.device)
    for i in range(2 * rh + 1):
        for j in range(2 * rw + 1):
            v = (v << 1) | (img[:, i:i + h - 2 * rh, j:j + w - 2 * rw] < c).long()
    out[:, rh:h - rh, rw:w - rw] = v
    return out


def _popcount(v):
    """Set bits of non-negative int64 values."""
    v = v - ((v >> 1) & 0x5555555555555555)
    v = (v & 0x3333333333333333) + ((v >> 2) & 0x3333333333333333)
    v = (v + (v >> 4)) & 0x0F0F0F0F0F0F0F0F
    v = v + (v >> 8)
    v = v + (v >> 16)
    return (v + (v >> 32)) & 0x7F


def _cost(base, match, min_d, d, l2r, cs, l2r_cost=None):
    """Hamming cost [n, h, w, d] uint8; partner columns outside the image
    use column 0; the 5x5 right view keeps the left view's cost at the last
    pixel of every d-pixel block."""
    n, h, w = base.shape
    x = torch.arange(w, device=base.device)
    out = torch.empty(n, h, w, d, dtype=torch.uint8, device=base.device)
    for t in range(d):
        xm = x - min_d - t if l2r else x + min_d + t
        xm = torch.where((xm >= 0) & (xm < w), xm, 0)
        out[..., t] = _popcount(base ^ match[:, :, xm]).to(torch.uint8)
    if not l2r and cs == 0:
        x0 = max(0, min_d)
        skip = (x >= x0) & (((x - x0) % d == d - 1) | (x == w - 1))
        out[:, :, skip] = l2r_cost[:, :, skip]
    return out


def _aggregate_sum(cost, x0, p1, p2):
    """Sum of the four stored path costs, int16 [n, h, w, d]."""
    n, h, w, d = cost.shape
    total = torch.zeros(n, h, w, d, dtype=torch.int16, device=cost.device)
    for axis, lo, hi in ((2, x0, w), (1, 0, h)):
        lines = h if axis == 2 else w
        pad = torch.full((2 * n, lines, d + 2), 127, dtype=torch.int32, device=cost.device)
        last = None
        for i in range(hi - lo):
            a, b = lo + i, hi - 1 - i
            c = torch.cat([cost.select(axis, a), cost.select(axis, b)]).int()
            if last is not None:
                m = last.amin(-1, keepdim=True)
                pad[..., 1:-1] = last + p1
                v = torch.minimum(torch.minimum(pad[..., :-2], pad[..., 2:]), torch.minimum(last, m + p2))
                c = c + v - m
            last = c
            stored = (c & 255).to(torch.int16)
            total.select(axis, a).add_(stored[:n])
            total.select(axis, b).add_(stored[n:])
    return total


def _wta(total, x0, y_rows, lo_ok, hi_ok, edge_c3, offset, uniq):
    """Winner, uniqueness and parabola of summed costs: float64 [h, w].
    lo_ok..hi_ok: winners kept; edge_c3: the right neighbour of winner d - 1;
    offset: disparity of index 0, a number or a [h, w] tensor."""
    h, w, d = total.shape
    out = torch.full((h, w), INVALID, dtype=torch.float64, device=total.device)
    y1, x1 = min(y_rows, h - 4), w - 4
    xs = max(5, x0)
    if y1 <= 5 or x1 <= xs:
        return out
    ids = torch.arange(d, device=total.device, dtype=torch.int32)
    rows = max(1, (1 << 27) // (w * d))
    for y in range(5, y1, rows):
        ye = min(y + rows, y1)
        s = total[y:ye, xs:x1].int()
        key = (s * 1024 + ids).amin(-1)
        ds, c2 = (key & 1023).long(), (key >> 10).double()
        c1 = s.gather(-1, (ds - 1).clamp(min=0)[..., None])[..., 0].double()
        c3 = s.gather(-1, (ds + 1).clamp(max=d - 1)[..., None])[..., 0].double()
        c3 = torch.where(ds == d - 1, float(edge_c3), c3)
        off = offset[y:ye, xs:x1] if torch.is_tensor(offset) else offset
        keep = (ds >= lo_ok) & (ds <= hi_ok) & ~(torch.minimum(c1 - c2, c3 - c2) <= c2 * (1.0 - uniq))
        den = (c1 + c3 - 2 * c2).clamp(min=1.0)
        out[y:ye, xs:x1] = torch.where(keep, (ds + off).double() + (c1 - c3 + den) / (2 * den), INVALID)
    return out


def _lr_check(dl, dr, thr=1.0):
    h, w = dl.shape
    x = torch.arange(w, device=dl.device, dtype=torch.float64)
    xr = (torch.where(x - dl > 0, x - dl + 0.5, x - dl - 0.5)).trunc().long()
    valid = dl != INVALID
    inside = valid & (xr >= 0) & (xr < w)
    xr = xr.clamp(0, w - 1)
    partner = dr.gather(1, xr)
    bad = inside & ((dl - partner).abs() > thr)
    out = torch.where(inside & ~bad, (dl + partner) / 2, INVALID)
    right = dr.clone().view(-1)
    rows = torch.arange(h, device=dl.device)[:, None] * w
    right[(rows + xr)[bad]] = INVALID
    return out, right.view(h, w)


def _median(m):
    h, w = m.shape
    p = torch.full((h + 2, w + 2), INVALID, dtype=m.dtype, device=m.device)
    p[1:-1, 1:-1] = m
    win = torch.stack([p[i:i + h, j:j + w] for i in range(3) for j in range(3)])
    out = win.sort(0).values[4]
    out[0], out[:, 0] = m[0], m[:, 0]
    return out


def _match(left, right, min_d, d, cs, p1, p2, uniq):
    """Left and right maps [n, h, w] float64 of pairs [n, h, w], LR check and
    median on."""
    n, h, w = left.shape
    x0 = max(0, min_d)
    cl, cr = _census(left, cs, False), _census(right, cs, True)
    cost = _cost(cl, cr, min_d, d, True, cs)
    cost = torch.cat([cost, _cost(cr, cl, min_d, d, False, cs, cost)])
    total = _aggregate_sum(cost, x0, p1, p2)
    two_row = d in (64, 128)
    maps = [_wta(total[k], x0, 2 * (h // 2) if two_row else h, 1, d - 1 if two_row else d - 2, d - 1,
                 min_d, uniq) for k in range(2 * n)]
    checked = [_lr_check(maps[k], maps[n + k]) for k in range(n)]
    return [_median(c[0]) for c in checked], [c[1] for c in checked]


def _interval(case):
    span, r = case["max_disp"] // (1 << (case["layers"] - 1)), 64
    while r < span:
        r *= 2
    return r // 2 if r > 2 * case["w"] else r


def _dilate(m):
    h, w = m.shape
    s = min(h, w)
    r = 1 if s < 360 else 2 if s < 720 else 3
    out = m.clone()
    if h > 2 * r + 1 and w > 2 * r + 1:
        mx = torch.nn.functional.max_pool2d(m[None, None], 2 * r + 1, 1)[0, 0]
        core = m[r + 1:h - r, r + 1:w - r]
        out[r + 1:h - r, r + 1:w - r] = torch.where(core == INVALID, mx[1:, 1:], core)
    return out


def _remove_peaks(m, ratio):
    """Segments (4-neighbours within 1.0) below the size threshold become invalid."""
    h, w = m.shape
    valid = m != INVALID
    label = torch.arange(h * w, device=m.device).view(h, w)
    # joins are decided on the float32 map the removal is given
    f = m.float()
    jh = valid[:, 1:] & valid[:, :-1] & ((f[:, 1:] - f[:, :-1]).abs() <= 1)
    jv = valid[1:] & valid[:-1] & ((f[1:] - f[:-1]).abs() <= 1)
    while True:
        new = label.clone()
        for a, b, j in ((new[:, 1:], new[:, :-1], jh), (new[1:], new[:-1], jv)):
            low = torch.minimum(a, b)
            a.copy_(torch.where(j, low, a))
            b.copy_(torch.where(j, torch.minimum(low, b), b))
        flat = new.view(-1)
        # labels only fall: follow them to their own labels, then hand each
        # segment's lowest back to the pixels named by the old labels
        root = torch.arange(h * w, device=m.device).scatter_reduce(0, label.view(-1), flat, "amin")
        flat = torch.minimum(flat, root[flat])
        flat = torch.minimum(flat, flat[flat])
        new = flat.view(h, w)
        if torch.equal(new, label):
            break
        label = new
    size = torch.bincount(label.view(-1), minlength=h * w)[label]
    least = int(np.float32(w * h) * np.float32(ratio))
    return torch.where(valid & (size < least), INVALID, m)


def _window_level(left, right, coarse, window, cs, p1, p2, uniq):
    """One finer level around twice the coarse map: float64 [h, w]."""
    h, w = left.shape
    dev = left.device
    # base disparities: even rows from the coarse map, odd and last rows copy
    cx = (torch.arange(w, device=dev) >> 1).clamp(max=w // 2 - 1)
    row = torch.arange(h, device=dev)
    row = torch.where((row % 2 == 1) | (row == h - 1), row - 1, row)
    row = torch.where(row % 2 == 1, row - 1, row)
    src = coarse[row >> 1][:, cx]
    bad = src == INVALID
    b = torch.where(bad, -32768, (2 * src.float() - window // 2).trunc().long())
    cl, cr = _census(left[None], cs, False)[0], _census(right[None], cs, True)[0]
    x = torch.arange(w, device=dev)
    half = window // 2
    table = (1, 2, 7, 20, 54)
    cost = torch.empty(h, w, window, dtype=torch.uint8, device=dev)
    for t in range(window):
        xr = x - t - b
        inside = (xr > 0) & (xr < w)
        c = _popcount(cl ^ cr.gather(1, xr.clamp(0, w - 1))) + table[min(4, 4 * abs(t - half) // half)]
        cost[..., t] = torch.where(inside, c, 255 if cs else 127).to(torch.uint8)
    total = torch.zeros(h, w, window, dtype=torch.int16, device=dev)
    t_ids = torch.arange(window, device=dev)
    for axis, n in ((1, w), (0, h)):
        line_b = torch.stack([b.select(axis, 0), b.select(axis, n - 1 if axis == 1 else 0)])
        last = torch.stack([cost.select(axis, 0), cost.select(axis, n - 1)]).long()
        total.select(axis, 0).add_(last[0].to(torch.int16))
        total.select(axis, n - 1).add_(last[1].to(torch.int16))
        m = last.amin(-1, keepdim=True)
        prev = line_b[..., None]
        for i in range(1, n):
            pa, pb = i, n - 1 - i
            bb = torch.stack([b.select(axis, pa), b.select(axis, pb)])[..., None]
            c = torch.stack([cost.select(axis, pa), cost.select(axis, pb)]).long()
            ok = bb != -32768
            shift = bb - prev
            pen = torch.clamp(p2 // (shift - 1).abs().clamp(min=1), min=p1)

            def side(k):
                idx = t_ids + shift + k
                got = last.gather(-1, idx.clamp(0, window - 1)) + p1
                return torch.where((idx >= 0) & (idx < window), got & 0xFFFFFFFF, 127)

            v = torch.minimum(torch.minimum(side(-1), side(1)),
                              torch.minimum(last, (m + pen) & 0xFFFFFFFF))
            new = (c + v - m) & 0xFFFFFFFF
            m = torch.where(ok, new.amin(-1, keepdim=True), 127)
            last = torch.where(ok, new, last)
            prev = torch.where(ok, bb, prev)
            stored = torch.where(ok, new & 255, 0).to(torch.int16)
            total.select(axis, pa).add_(stored[0])
            total.select(axis, pb).add_(stored[1])
    out = _wta(total, 0, 4 * (h // 4), 2, window - 2, 0, b, uniq)
    return _median(torch.where(bad, INVALID, out))


def _pyramid(case, left, right, window, cs, p1, p2, peaks):
    layers = case["layers"]
    ls, rs = [left], [right]
    for _ in range(layers - 1):
        h, w = ls[-1].shape
        ls.append(ls[-1][:h // 2 * 2:2, :w // 2 * 2:2].contiguous())
        rs.append(rs[-1][:h // 2 * 2:2, :w // 2 * 2:2].contiguous())
    d = _interval(case)
    cur = _match(ls[-1][None], rs[-1][None], 0, d, cs, p1, p2, 0.95 if layers == 1 else 1.0)[0][0]
    if layers > 1:
        cur = _dilate(cur)
    if peaks:
        cur = _remove_peaks(cur, {1: 0.0005, 2: 0.001}.get(layers, 0.005))
    for i in range(layers - 2, -1, -1):
        cur = _window_level(ls[i], rs[i], cur, window, cs, p1, p2, 0.95 if i == 0 else 1.0)
    return cur


def _diff_exact(cost, p1, p2, up):
    """Forward and backward of the differentiable form in float64, the first
    of equal candidates in the order (d, d - 1, d + 1, minimum) winning."""
    c, q1, q2, g = (t.detach().double() for t in (cost, p1, p2, up))
    n, h, w, d = c.shape
    ids = torch.arange(d, device=c.device)
    total = torch.zeros_like(c)
    record = []
    inf = float("inf")
    for axis in (2, 1):
        steps = w if axis == 2 else h
        lines = h if axis == 2 else w
        for back in (False, True):
            order = list(range(steps))[::-1] if back else list(range(steps))
            win = torch.zeros(steps, n, lines, d, dtype=torch.uint8, device=c.device)
            arg = torch.zeros(steps, n, lines, 1, dtype=torch.long, device=c.device)
            pad = torch.full((n, lines, d + 2), inf, dtype=torch.float64, device=c.device)
            last = None
            for s, i in enumerate(order):
                cur = c.select(axis, i)
                if last is not None:
                    m = last.amin(-1, keepdim=True)
                    arg[s] = torch.where(last == m, ids, d).amin(-1, keepdim=True)
                    pad[..., 1:-1] = last
                    a = q1.select(axis, i)[..., None]
                    best, code = last, win[s]
                    for k, cand in ((1, pad[..., :-2] + a), (2, pad[..., 2:] + a),
                                    (3, m + q2.select(axis, i)[..., None])):
                        less = cand < best
                        code.masked_fill_(less, k)
                        best = torch.where(less, cand, best)
                    cur = cur + best - m
                last = cur
                total.select(axis, i).add_(cur)
            record.append((axis, order, win, arg))
    e = torch.softmax(-total / TEMPERATURE, -1)
    disp = (e * ids).sum(-1)
    gs = g[..., None] * (-1.0 / TEMPERATURE) * e * (ids - disp[..., None])
    del e, total
    gc, g1, g2 = torch.zeros_like(c), torch.zeros_like(q1), torch.zeros_like(q2)
    for axis, order, win, arg in record:
        grad = gs.select(axis, order[-1]).clone()
        for s in range(len(order) - 1, -1, -1):
            i = order[s]
            gc.select(axis, i).add_(grad)
            if s == 0:
                break
            code = win[s]
            stay, below, above = ((grad * (code == k) for k in (0, 1, 2)))
            least = (grad * (code == 3)).sum(-1, keepdim=True)
            g1.select(axis, i).add_((below + above).sum(-1))
            g2.select(axis, i).add_(least[..., 0])
            prev = gs.select(axis, order[s - 1]) + stay
            prev[..., :-1] += below[..., 1:]
            prev[..., 1:] += above[..., :-1]
            prev.scatter_add_(-1, arg[s], least - grad.sum(-1, keepdim=True))
            grad = prev
    return disp, gc, g1, g2


def exact(case, seed):
    k = case["kind"]
    if k == "diff":
        return _diff_exact(*_diff_inputs(case, seed))
    images = _images(case, seed)
    if k in ("pair", "pair_host"):
        (left, right), = images
        dl, dr = _match(left[None], right[None], case["min_d"], case["d"], case["cs"], case["p1"],
                        case["p2"], 0.95)
        return [dl[0], dr[0]] if case["right"] else [dl[0]]
    if k == "batch":
        left, right = (torch.stack(t) for t in zip(*images))
        return _match(left, right, 0, case["d"], 1, 10, 150, 0.95)[0]
    if k == "uneven":
        return [_match(a[None], b[None], 0, d, 1, 10, 150, 0.95)[0][0]
                for (a, b), (_, _, d) in zip(images, _mix(case))]
    (left, right), = images
    if k == "pyramid":
        return _pyramid(case, left, right, case["window"], 1, 10, 150, False)
    return _pyramid(case, left, right, FasterStereoCuda.LEVEL_RANGE, 0, 8, 32, True)
