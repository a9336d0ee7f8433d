"""Timed cases of the geodesic distance transforms.

Each case is one call that a program makes through the package's public entry
points: plain 2D and 3D calls (unsigned, signed, geodesic symmetric filtering)
and batched calls.  `listed()` names the fixed cases, `draw(rng)` gives one
more case from the same ranges:

  2D     sides 64 to 2048, 1 or 3 channels, iter 2 to 4
  3D     sides 16 to 512 (at most 512^3 voxels x 4 iterations x transforms),
         1 or 2 channels, spacing 0.5 to 3, iter 2 to 4
  batch  16 to 64 uneven images and volumes in one call
  clicks 2 to 16 resident volumes, one signed transform each, in one call,
         with the transposed images that such a program keeps

The transforms keep the two roundings of every candidate of the reference's
CPU path, so another correct implementation returns the same bits:
`tolerance` is "exact".  `exact` computes the same raster passes in 64 bits.
"""
import math
import random

import torch

import fastgeodis_amd as FG

TRANSFORMS = {"unsigned": 1, "signed": 2, "gsf": 6}


# ---- the cases ---------------------------------------------------------------

def _case2d(op, H, W, C=1, lamb=1.0, iters=2, v=1e10, theta=0.0):
    return {"kind": "2d", "op": op, "C": C, "D": 1, "H": H, "W": W, "lamb": lamb, "iter": iters, "v": v,
            "theta": theta}


def _case3d(op, D, H, W, C=1, lamb=1.0, iters=4, v=1e10, theta=0.0, spacing=(1.0, 1.0, 1.0)):
    return {"kind": "3d", "op": op, "C": C, "D": D, "H": H, "W": W, "lamb": lamb, "iter": iters, "v": v,
            "theta": theta, "s_d": spacing[0], "s_h": spacing[1], "s_w": spacing[2]}


def listed():
    cases = [
        # the smallest image of the published speed comparison: launches and latency
        ("2d_64", _case2d("unsigned", 64, 64)),
        # the published 512^2 comparison: one grey image, one call
        ("2d_512", _case2d("unsigned", 512, 512)),
        # a signed distance (both sides of an outline) of an odd-sized photograph
        ("2d_signed_481x723", _case2d("signed", 481, 723, C=3, lamb=0.5)),
        # the colour photograph of the 2D demonstration, mixed distance
        ("2d_rgb_1536", _case2d("unsigned", 1536, 1536, C=3, lamb=0.5)),
        # smoothing a noisy segmentation, as the 2D filtering demonstration does
        ("2d_gsf_1252x1292", _case2d("gsf", 1252, 1292, v=1000.0, theta=0.1)),
        # the small crop of the 3D demonstration
        ("3d_crop_20x120x140", _case3d("unsigned", 20, 120, 140)),
        # an anisotropic scan, mixed distance, default iterations
        ("3d_128x256x256", _case3d("unsigned", 128, 256, 256, lamb=0.5, spacing=(2.5, 1.0, 1.0))),
        # signed distance to an outline in the same scan, pure geodesic
        ("3d_signed_128x256x256", _case3d("signed", 128, 256, 256, spacing=(2.5, 1.0, 1.0))),
        # two registered modalities on an odd grid
        ("3d_2ch_97x211x163", _case3d("unsigned", 97, 211, 163, C=2, lamb=0.8, spacing=(2.1, 0.9, 0.9))),
        # the published 512^3 comparison at the default iterations
        ("3d_512", _case3d("unsigned", 512, 512, 512)),
        # a data-loading step: uneven images and volumes in one call
        ("batch_48_8", {"kind": "batch", "n2d": 48, "n3d": 8, "sizes": 4, "lamb": 1.0, "iter": 2, "v": 1e10}),
        # interactive segmentation: a click each in eight resident volumes
        ("clicks_8", {"kind": "clicks", "n": 8, "lo": 96, "hi": 320, "sizes": 5, "lamb": 1.0, "iter": 2, "v": 1e10}),
    ]
    return [dict(c, name=name) for name, c in cases]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = work(_case3d("unsigned", 512, 512, 512))
    while True:
        kind = rng.choice(["2d", "2d", "2d", "3d", "3d", "3d", "batch", "clicks"])
        op = rng.choice(["unsigned", "unsigned", "signed", "gsf"])
        lamb = rng.choice([1.0, 1.0, 0.5, 0.0, round(rng.uniform(0.05, 0.95), 2)])
        iters = rng.choice([2, 2, 4])
        if kind == "2d":
            c = _case2d(op, _log_int(rng, 64, 2048), _log_int(rng, 64, 2048), rng.choice([1, 3]), lamb, iters,
                        rng.choice([1e10, 1000.0]), 0.1 if op == "gsf" else 0.0)
        elif kind == "3d":
            c = _case3d(op, _log_int(rng, 16, 512), _log_int(rng, 32, 512), _log_int(rng, 32, 512),
                        rng.choice([1, 1, 2]), lamb, iters, 1e10, 0.1 if op == "gsf" else 0.0,
                        tuple(round(rng.uniform(0.5, 3.0), 2) for _ in range(3)))
        elif kind == "batch":
            c = {"kind": "batch", "n2d": rng.randint(12, 56), "n3d": rng.randint(4, 8),
                 "sizes": rng.randrange(1 << 20), "lamb": lamb, "iter": 2, "v": 1e10}
        else:
            lo = rng.randint(64, 160)
            c = {"kind": "clicks", "n": rng.randint(2, 16), "lo": lo, "hi": rng.randint(lo + 16, 320),
                 "sizes": rng.randrange(1 << 20), "lamb": 1.0, "iter": 2, "v": 1e10}
        w = work(c)
        if w["flops"] <= most["flops"] and w["bytes"] <= most["bytes"]:
            return c


def _members(case):
    """(kind, op, C, shape, spacing) of each instance of a case."""
    if case["kind"] in ("2d", "3d"):
        shape = (case["H"], case["W"]) if case["kind"] == "2d" else (case["D"], case["H"], case["W"])
        sp = None if case["kind"] == "2d" else [case["s_d"], case["s_h"], case["s_w"]]
        return [(case["kind"], case["op"], case["C"], shape, sp)]
    rng = random.Random(case["sizes"])
    out = []
    if case["kind"] == "clicks":
        for _ in range(case["n"]):
            shape = tuple(rng.randint(case["lo"], case["hi"]) for _ in range(3))
            out.append(("3d", "signed", 1, shape, [2.0, 1.0, 1.0]))
        return out
    for _ in range(case["n2d"]):
        shape = (_log_int(rng, 64, 2048), _log_int(rng, 64, 2048))
        out.append(("2d", "unsigned", rng.choice([1, 3]), shape, None))
    for _ in range(case["n3d"]):
        shape = tuple(rng.randint(64, 256) for _ in range(3))
        out.append(("3d", "unsigned", 1, shape, [round(rng.uniform(0.5, 3.0), 2) for _ in range(3)]))
    return out


# ---- inputs and the call -----------------------------------------------------

def _image(shape, C, rng, gen):
    """(1, C, *shape): blobs of several widths plus a little noise, like a smooth scan or photograph."""
    img = 0.05 * torch.rand((1, C, *shape), generator=gen, device="cuda")
    axes = [torch.arange(s, dtype=torch.float32, device="cuda") for s in shape]
    for c in range(C):
        for _ in range(10):
            width = rng.uniform(8.0, 60.0)
            prof = [torch.exp(-((a - rng.uniform(0, s)) ** 2) / (2 * width * width)) for a, s in zip(axes, shape)]
            prof[0] *= rng.uniform(0.1, 1.0)
            blob = prof[0]
            for p in prof[1:]:
                blob = blob.unsqueeze(-1) * p
            img[0, c] += blob
    return img


def _mask(op, shape, clicked, rng, gen):
    if clicked:  # 0.5 everywhere, object clicks 1, background clicks 0
        m = torch.full(shape, 0.5, device="cuda")
        for k in range(rng.randint(2, 6)):
            m[tuple(rng.randrange(s) for s in shape)] = 1.0 if k % 2 == 0 else 0.0
    elif op == "unsigned":  # ones with a few seeds
        m = torch.ones(shape, device="cuda")
        for _ in range(rng.randint(2, 16)):
            m[tuple(rng.randrange(s) for s in shape)] = 0.0
    else:  # a filled ellipsoid; the filter's input has 2 % of its elements flipped
        r2 = None
        for k, s in enumerate(shape):
            a = torch.arange(s, dtype=torch.float32, device="cuda")
            q = ((a - rng.uniform(0.35, 0.65) * s) / (rng.uniform(0.15, 0.3) * s)) ** 2
            r2 = q if r2 is None else r2.unsqueeze(-1) + q
        m = (r2 > 1.0).float()
        if op == "gsf":
            m = torch.where(torch.rand(shape, generator=gen, device="cuda") < 0.02, 1.0 - m, m)
    return m[None, None].contiguous()


def prepare(case, seed):
    rng = random.Random(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = {"case": case, "items": []}
    for kind, op, C, shape, sp in _members(case):
        clicked = case["kind"] == "clicks"
        img = _image(shape, C, rng, gen)
        state["items"].append((kind, op, img, _mask(op, shape, clicked, rng, gen), sp))
    if case["kind"] in ("batch", "clicks"):
        state["instances"] = [
            FG.Instance(img, mask, case["v"], case["lamb"], iter=case["iter"], spacing=sp, op=op,
                        image_t=FG.transposed_image(img) if case["kind"] == "clicks" else None)
            for _, op, img, mask, sp in state["items"]]
    return state


def run(state):
    case = state["case"]
    if case["kind"] in ("batch", "clicks"):
        return FG.geodesic_batch(state["instances"])
    kind, op, img, mask, sp = state["items"][0]
    v, lamb, iters, theta = case["v"], case["lamb"], case["iter"], case["theta"]
    if kind == "2d":
        if op == "unsigned":
            return FG.generalised_geodesic2d(img, mask, v, lamb, iters)
        if op == "signed":
            return FG.signed_generalised_geodesic2d(img, mask, v, lamb, iters)
        return FG.GSF2d(img, mask, theta, v, lamb, iters)
    if op == "unsigned":
        return FG.generalised_geodesic3d(img, mask, sp, v, lamb, iters)
    if op == "signed":
        return FG.signed_generalised_geodesic3d(img, mask, sp, v, lamb, iters)
    return FG.GSF3d(img, mask, theta, sp, v, lamb, iters)


def work(case):
    """Image and mask read once and the result written once; the operations of
    every neighbour candidate (difference, weight, sums, minimum)."""
    nbytes, flops = 0.0, 0.0
    for kind, op, C, shape, _ in _members(case):
        n = float(math.prod(shape))
        nbytes += n * (4 * C + 8)
        per = (3 if case["lamb"] == 1.0 else 5) + 2 * (C - 1)
        sweeps, cand = (4, 3) if kind == "2d" else (6, 9)
        flops += n * sweeps * case["iter"] * TRANSFORMS[op] * cand * per
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    return "exact"


# ---- the same passes in 64 bits ----------------------------------------------

def _sweep(img, d, axis, le, lg, table, outside):
    """One pass pair along spatial axis `axis` of img (B, C, *S) and d (B, *S),
    in place; table: (B, 3, ...) steps to the previous slice's neighbours;
    outside: None or the elements that only pad a smaller image, which stay
    unreachable."""
    nd = d.dim() - 1
    img, d = img.movedim(2 + axis, 0), d.movedim(1 + axis, 0)  # (A, B, C, *plane), (A, B, *plane)
    outside = None if outside is None else outside.movedim(1 + axis, 0)
    n = d.shape[0]
    inf = float("inf")
    pad = (1, 1) * (nd - 1)
    step = (le * table).reshape(table.shape[0], *([1] * (nd - 1)), *table.shape[1:])
    for order in (range(1, n), range(n - 2, -1, -1)):
        back = -1 if order.step > 0 else 1
        for a in order:
            dq = torch.nn.functional.pad(d[a + back], pad, value=inf)
            iq = torch.nn.functional.pad(img[a + back], pad)
            for k in range(nd - 1):
                dq, iq = dq.unfold(1 + k, 3, 1), iq.unfold(2 + k, 3, 1)
            here = img[a].reshape(*img[a].shape, *([1] * (nd - 1)))
            cand = dq + step + lg * (iq - here).abs().sum(1)
            new = torch.minimum(d[a], cand.flatten(-(nd - 1)).amin(-1))
            d[a] = new if outside is None else new.masked_fill_(outside[a], inf)


def _transform(img, d, spacings, lamb, iters, outside=None):
    """The raster passes of a batch img (B, C, *S), d (B, *S); spacings: per instance (3D)."""
    nd, B = d.dim() - 1, d.shape[0]
    tables = []
    if nd == 2:
        row = torch.tensor([math.sqrt(2.0), 1.0, math.sqrt(2.0)], dtype=torch.float64, device=d.device)
        tables = [row.expand(B, 3)] * 2
    else:
        s = torch.tensor(spacings, dtype=torch.float64, device=d.device) ** 2
        off = torch.tensor([1.0, 0.0, 1.0], dtype=torch.float64, device=d.device)
        for axis in range(3):
            b, e = [k for k in range(3) if k != axis]
            tables.append((s[:, axis, None, None] + s[:, b, None, None] * off[:, None] + s[:, e, None, None] * off).sqrt())
    for _ in range(iters):
        for axis in range(nd):
            _sweep(img, d, axis, 1.0 - lamb, lamb, tables[axis], outside)
    return d


def _apply(op, img, mask, spacings, case):
    v, lamb, iters = case["v"], case["lamb"], case["iter"]

    def dist(m):
        return _transform(img, v * m, spacings, lamb, iters)

    def signed(m):
        return dist(m) - dist(1.0 - m)

    if op == "unsigned":
        return dist(mask)
    if op == "signed":
        return signed(mask)
    ds = signed(mask)
    md, me = (ds > case["theta"]).double(), (ds > -case["theta"]).double()
    return -signed(1.0 - md) + signed(me)


def exact(case, seed):
    items = prepare(case, seed)["items"]
    outs = [None] * len(items)
    flat = [i for i, it in enumerate(items) if it[0] == "2d"]
    if len(flat) > 1:  # images of a batch side by side, padded with unreachable elements
        C = max(items[i][2].shape[1] for i in flat)
        H, W = (max(items[i][2].shape[k] for i in flat) for k in (2, 3))
        img = torch.zeros((len(flat), C, H, W), dtype=torch.float64, device="cuda")
        d = torch.full((len(flat), H, W), float("inf"), dtype=torch.float64, device="cuda")
        for b, i in enumerate(flat):
            x, m = items[i][2][0].double(), items[i][3][0, 0].double()
            img[b, :x.shape[0], :x.shape[1], :x.shape[2]] = x
            d[b, :m.shape[0], :m.shape[1]] = case["v"] * m
        _transform(img, d, None, case["lamb"], case["iter"], torch.isinf(d))
        for b, i in enumerate(flat):
            h, w = items[i][3].shape[2:]
            outs[i] = d[b, :h, :w][None, None].clone()
    for i, (_, op, x, m, sp) in enumerate(items):
        if outs[i] is None:
            outs[i] = _apply(op, x.double(), m[0].double(), [sp], case)[None]
    return outs if case["kind"] in ("batch", "clicks") else outs[0]
