"""Performance cases of the operator path: what a program on these operators has the GPU do.

Each case is one call, or the short sequence of calls of one sample program, through
hipacc_amd.operators or hipacc_amd.autograd on prepared calls (descriptors and buffers a
program builds once and keeps), over the sizes of the samples, the tests and bench.py.
"""
import math

import numpy as np
import torch

from hipacc_amd import capi, masks
from hipacc_amd import operators as op

BOUNDARY = {"clamp": capi.CLAMP, "mirror": capi.MIRROR, "repeat": capi.REPEAT,
            "constant": capi.CONSTANT}
DTYPE = {"f32": torch.float32, "u8": torch.uint8}
BYTES = {"f32": 4, "u8": 1}
DEV = "cuda"


def listed():
    return [
        # the headline of bench.py: a 5x5 Gaussian over a large float image
        dict(name="conv5_f32_4096", kind="conv", dtype="f32", w=4096, h=4096, k=5,
             boundary="clamp"),
        # the smallest call in ordinary use: a thumbnail blurred in 8 bits, latency alone
        dict(name="conv3_u8_256", kind="conv", dtype="u8", w=256, h=256, k=3, boundary="clamp"),
        # the Sobel sample at its 12-megapixel photo: two integer derivatives and their magnitude
        dict(name="sobel_u8_4032x3024", kind="sobel", dtype="u8", w=4032, h=3024,
             boundary="clamp"),
        # separable Gaussian over a cropped float image: rows of odd length, no aligned rows
        dict(name="sep13_f32_2043x1531", kind="separable", dtype="f32", w=2043, h=1531, k=13,
             boundary="mirror"),
        # morphological opening (erode, dilate) of an 8-bit video frame
        dict(name="morph5_u8_1920x1080", kind="morph", dtype="u8", w=1920, h=1080, k=5,
             boundary="clamp"),
        # edge-preserving smoothing of a large float image, as bench.py runs it
        dict(name="bilateral13_f32_4096", kind="bilateral", dtype="f32", w=4096, h=4096, k=13,
             boundary="mirror"),
        # the Bilateral_Filter sample's 8-bit operator on a small odd-sized image
        dict(name="bilateral7_u8_1001x751", kind="bilateral", dtype="u8", w=1001, h=751, k=7,
             boundary="clamp"),
        # training step: learnable 9x9 mask, then 7x7 bilateral with learnable sigma,
        # forward and backward on a batch
        dict(name="train_16x1024", kind="train", dtype="f32", batch=16, w=1024, h=1024,
             boundary="clamp"),
        # Gaussian and Laplacian pyramids of a batch of uneven images
        dict(name="pyramid_32img_8lvl", kind="pyramid", dtype="f32", images=32, levels=8,
             w=4096, h=2160),
        # exposure statistics of a float image: sum, minimum, maximum and a 256-bin histogram
        dict(name="stats_f32_4096", kind="stats", dtype="f32", w=4096, h=4096),
        # the Mixed kernel-fusion sample: eight kernels as one launch
        dict(name="fused_mixed_f32_4096", kind="fused", dtype="f32", w=4096, h=4096,
             chain="PPLPPLPP", boundary="clamp"),
        # the Gaussian_Blur_RGBA sample on a video frame of uchar4 pixels
        dict(name="rgba5_u8_1920x1080", kind="rgba", dtype="u8", w=1920, h=1080, k=5,
             boundary="clamp"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["conv", "conv", "sobel", "separable", "morph", "bilateral", "bilateral",
                       "train", "pyramid", "stats", "fused", "rgba"])
    dtype = rng.choice(["f32", "u8"])
    boundary = rng.choice(sorted(BOUNDARY))
    # half of the widths are whole cache lines, as a padded allocation gives; the rest as they fall
    w, h = _log_int(rng, 100, 4096), _log_int(rng, 100, 4096)
    if rng.random() < 0.5:
        w = max(128, w // 64 * 64)
    c = dict(kind=kind, dtype=dtype, w=w, h=h)
    if kind in ("conv", "separable", "morph", "rgba", "bilateral"):
        sizes = {"conv": [3, 5, 7, 9], "separable": [3, 5, 7, 9, 13], "morph": [3, 5, 7],
                 "rgba": [3, 5, 7], "bilateral": [3, 5, 7, 9, 13]}
        c.update(k=rng.choice(sizes[kind]), boundary=boundary)
    if kind == "rgba":
        c.update(w=min(w, 2048))
    elif kind == "sobel":
        c.update(dtype="u8", boundary=boundary)
    elif kind == "train":
        c.update(dtype="f32", batch=rng.randint(1, 16), w=min(w, 1024), h=min(h, 1024),
                 boundary=boundary)
    elif kind == "pyramid":
        c.update(dtype="f32", images=rng.randint(1, 32), levels=rng.randint(3, 8),
                 w=max(w, 512), h=max(256, min(h, 2160)))
    elif kind == "fused":
        c.update(chain=rng.choice(["PL", "LP", "PLP", "LL", "PPLPPLPP"]), boundary=boundary)
    return c


# ---------------------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------------------
def _field(gen, *shape):
    """Photograph-like pixels in [0, 1]: a few low frequencies and sensor noise."""
    *lead, h, w = shape
    yy = torch.linspace(0, 1, h, device=DEV).view(h, 1)
    xx = torch.linspace(0, 1, w, device=DEV).view(1, w)
    out = torch.empty(shape, device=DEV)
    p = torch.rand((4, 4), generator=gen, device=DEV).tolist()
    f = torch.full((h, w), 0.5, device=DEV)
    for a, u, v, ph in p:
        f += 0.2 * a * torch.sin(2 * math.pi * ((1 + 7 * u) * xx + (1 + 7 * v) * yy + ph))
    out.copy_(f.expand(shape))
    out += 0.05 * torch.randn(shape, generator=gen, device=DEV)
    return out.clamp_(0.0, 1.0)


def _image(gen, dtype, *shape):
    f = _field(gen, *shape)
    return f if dtype == "f32" else (f * 255.0).round_().to(torch.uint8)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _pyramid_shapes(case):
    """(h, w) of the batch: the largest first, the others seeded by the case, not the run."""
    rng = np.random.default_rng(5005)
    n = case["images"]
    hs = rng.integers(256, case["h"] + 1, n) if case["h"] > 256 else np.full(n, case["h"])
    ws = rng.integers(256, case["w"] + 1, n)
    return [(case["h"], case["w"])] + [(int(a), int(b)) for a, b in zip(hs[1:], ws[1:])]


def _inputs(case, seed):
    g = _gen(seed)
    w, h, kind = case["w"], case["h"], case["kind"]
    if kind == "train":
        x = _field(g, case["batch"], h, w)
        wt = 0.1 * torch.randn((9, 9), generator=g, device=DEV)
        sigma = torch.full((1,), 0.1, device=DEV)
        gy = torch.randn(x.shape, generator=g, device=DEV)
        return x, wt, sigma, gy
    if kind == "pyramid":
        return [_field(g, a, b) for a, b in _pyramid_shapes(case)]
    if kind == "rgba":
        return _image(g, case["dtype"], h, 4 * w).view(h, w, 4)
    return _image(g, case["dtype"], h, w)


def _gauss(k):
    return masks.gaussian_2d(k, k / 5.0)


def _sep_taps(k):
    return masks.gaussian_1d(k, 3.0 if k == 13 else k / 4.0)


def _stages(case):
    """The fusion samples' kernels: P adds a constant, L is the 5x5 Gaussian."""
    dt = capi.F32 if case["dtype"] == "f32" else capi.U8
    beta = 0.25 if case["dtype"] == "f32" else 3.0
    cvt = capi.CVT_TRUNC if case["dtype"] == "f32" else capi.CVT_ROUND
    pt = dict(kind="point", dtype=dt, op=capi.POINT_AFFINE, alpha=1.0, beta=beta)
    lc = dict(kind="local", dtype=dt, mask_w=5, mask_h=5, weights=masks.gaussian_2d(5, 1.0),
              boundary=BOUNDARY[case["boundary"]], cvt=cvt)
    return [pt if ch == "P" else lc for ch in case["chain"]]


# ---------------------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------------------
def prepare(case, seed):
    kind, w, h = case["kind"], case["w"], case["h"]
    src = _inputs(case, seed)
    cvt = capi.CVT_ROUND if case["dtype"] == "u8" else capi.CVT_TRUNC
    bh = BOUNDARY.get(case.get("boundary"), capi.CLAMP)
    if kind == "train":
        x, wt, sigma, gy = src
        return dict(kind=kind, x=x.requires_grad_(), w=wt.requires_grad_(),
                    sigma=sigma.requires_grad_(), gy=gy, boundary=bh)
    if kind == "pyramid":
        return _prepare_pyramid(case, src)
    s = dict(kind=kind, src=src)
    if kind in ("conv", "separable", "bilateral", "fused", "rgba"):
        dst = torch.empty_like(src)
        s["out"] = [dst]
        if kind == "conv":
            call = op.prepare_local(src, dst, case["k"], case["k"], weights=_gauss(case["k"]),
                                    boundary=bh, cvt=cvt)
        elif kind == "separable":
            t = _sep_taps(case["k"])
            call = op.prepare_separable(src, dst, t, t, boundary=bh, cvt=cvt)
        elif kind == "bilateral":
            sr = 0.1 if case["dtype"] == "f32" else 25.0
            call = op.prepare_bilateral(src, dst, case["k"], case["k"] / 4.0, sr, boundary=bh,
                                        cvt=cvt)
        elif kind == "fused":
            call = op.prepare_fused(src, dst, _stages(case))
        else:
            dt = capi.U8X4 if case["dtype"] == "u8" else capi.F32X4
            call = op.prepare_local(src, dst, case["k"], case["k"], weights=_gauss(case["k"]),
                                    boundary=bh, cvt=cvt, src_dtype=dt, dst_dtype=dt)
        s["calls"] = [call]
    elif kind == "sobel":
        dx = torch.empty((h, w), dtype=torch.int16, device=DEV)
        dy, mag = torch.empty_like(dx), torch.empty_like(src)
        sx, sy = masks.SOBEL_X, masks.SOBEL_Y
        s["calls"] = [
            op.prepare_local(src, dx, 3, 3, weights=sx, domain=(sx != 0).astype(np.uint8),
                             acc_float=False, boundary=bh),
            op.prepare_local(src, dy, 3, 3, weights=sy, domain=(sy != 0).astype(np.uint8),
                             acc_float=False, boundary=bh),
            op.prepare_point(capi.POINT_MAGNITUDE, dx, mag, dy, alpha=4.0)]
        s["out"] = [dx, dy, mag]
    elif kind == "morph":
        ero, opened = torch.empty_like(src), torch.empty_like(src)
        f = case["dtype"] == "f32"
        s["calls"] = [op.prepare_local(src, ero, case["k"], case["k"], reduce=capi.MIN,
                                       acc_float=f, boundary=bh),
                      op.prepare_local(ero, opened, case["k"], case["k"], reduce=capi.MAX,
                                       acc_float=f, boundary=bh)]
        s["out"] = [ero, opened]
    elif kind == "stats":
        f = case["dtype"] == "f32"
        red = [torch.zeros(1, dtype=torch.float32 if f else torch.int32, device=DEV)
               for _ in range(3)]
        bins = torch.zeros(256, dtype=torch.int32, device=DEV)
        s["calls"] = [op.ReduceCall(src, m, r) for m, r in zip((capi.SUM, capi.MIN, capi.MAX), red)]
        s["calls"].append(op.HistogramCall(src, 256, bins, scale=256.0 if f else 1.0))
        s["out"] = red + [bins]
    return s


def _prepare_pyramid(case, images):
    """All levels of the batch in two arenas, each level a contiguous image on a 512-byte line."""
    levels = case["levels"]

    def carve(first):
        spots, n = [], 0
        for im in images:
            h, w = im.shape
            spots.append([])
            for l in range(first, levels if first else levels - 1):
                spots[-1].append((n, h >> l, w >> l))
                n += ((h >> l) * (w >> l) + 127) // 128 * 128
        arena = torch.zeros(n, device=DEV)
        return arena, [[arena[o:o + a * b].view(a, b) for o, a, b in row] for row in spots]

    ga, gs = carve(1)
    la, ls = carve(0)
    plan = op.PyramidPlan([[im] + row for im, row in zip(images, gs)], ls)
    return dict(kind="pyramid", plan=plan, out=[ga, la], keep=images)


def run(state):
    kind = state["kind"]
    if kind == "train":
        from hipacc_amd import autograd as ag
        b = state["boundary"]
        y = ag.bilateral(ag.conv2d(state["x"], state["w"], b), state["sigma"], 7, 2.0, b)
        gx, gw, gs = torch.autograd.grad(y, (state["x"], state["w"], state["sigma"]), state["gy"])
        return [y, gx, gw, gs]
    if kind == "pyramid":
        state["plan"].run()
    else:
        for call in state["calls"]:
            call.launch()
    return state["out"]


def work(case):
    kind, n = case["kind"], case["w"] * case["h"]
    e = BYTES[case["dtype"]]
    k2 = case.get("k", 0) ** 2
    if kind == "conv":
        return dict(bytes=2 * e * n, flops=2 * k2 * n)
    if kind == "separable":
        return dict(bytes=2 * e * n, flops=4 * case["k"] * n)
    if kind == "rgba":
        return dict(bytes=8 * e * n, flops=8 * k2 * n)
    if kind == "sobel":   # image in; dx, dy (16 bits each) and magnitude out
        return dict(bytes=6 * n, flops=(2 * 2 * 6 + 6) * n)
    if kind == "morph":   # image in, eroded and opened image out; separable comparisons
        return dict(bytes=3 * e * n, flops=4 * (case["k"] - 1) * n)
    if kind == "bilateral":   # per tap: difference, square, scale, add, exponential, 3 of the sums
        return dict(bytes=2 * e * n, flops=8 * k2 * n)
    if kind == "fused":
        return dict(bytes=2 * e * n, flops=sum(50 if c == "L" else 2 for c in case["chain"]) * n)
    if kind == "stats":
        return dict(bytes=e * n, flops=5 * n)
    if kind == "train":   # x, gy in; y, gx out; three 9x9 products, bilateral and its adjoint
        n *= case["batch"]
        return dict(bytes=16 * n, flops=(6 * 81 + 28 * 49) * n)
    px = [a * b for a, b in _pyramid_shapes(case)]
    n0 = sum(px)
    below = sum((a >> l) * (b >> l) for a, b in _pyramid_shapes(case)
                for l in range(1, case["levels"]))
    above = sum((a >> l) * (b >> l) for a, b in _pyramid_shapes(case)
                for l in range(case["levels"] - 1))
    return dict(bytes=4 * (n0 + below + above), flops=50 * below + 12 * above)


# ---------------------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------------------
def _index(n, r, boundary):
    """Source index of each position -r .. n+r-1, and whether it is outside the image."""
    i = torch.arange(-r, n + r, device=DEV)
    outside = (i < 0) | (i >= n)
    if boundary == capi.REPEAT:
        j = i % n
    elif boundary == capi.MIRROR:
        j = torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))
    else:
        j = i
    return j.clamp(0, n - 1), outside


def _pad(x, ry, rx, boundary):
    """x with its boundary handling applied r pixels beyond each edge (constant: 0)."""
    jy, oy = _index(x.shape[-2], ry, boundary)
    jx, ox = _index(x.shape[-1], rx, boundary)
    p = x[..., jy, :][..., jx]
    if boundary == capi.CONSTANT:
        p = p.masked_fill(oy[:, None] | ox[None, :], 0.0)
    return p


def _conv64(x, w, boundary):
    kh, kw = w.shape
    h, wd = x.shape[-2:]
    p = _pad(x, kh // 2, kw // 2, boundary)
    y = torch.zeros_like(x)
    for dy in range(kh):
        for dx in range(kw):
            y = y + w[dy, dx] * p[..., dy:dy + h, dx:dx + wd]
    return y


def _bilateral64(x, k, sigma_d, sigma_r, boundary):
    r = k // 2
    h, wd = x.shape[-2:]
    p = _pad(x, r, r, boundary)
    num, den = torch.zeros_like(x), torch.zeros_like(x)
    for dy in range(k):
        for dx in range(k):
            v = p[..., dy:dy + h, dx:dx + wd]
            sp = math.exp(-((dx - r) ** 2 + (dy - r) ** 2) / (2.0 * sigma_d * sigma_d))
            s = torch.exp(-(v - x) ** 2 / (2.0 * sigma_r ** 2)) * sp
            num = num + s * v
            den = den + s
    return num / den


def _map(src, dst):
    """Interpolation's mapped positions: defined in float, whatever the pixels are."""
    s = np.float32(src) / np.float32(dst)
    return (s / np.float32(2)) + s * np.arange(dst, dtype=np.float32)


def _pyramid64(case, images):
    w5 = torch.tensor([1.0, 4.0, 6.0, 4.0, 1.0], dtype=torch.float64, device=DEV)
    w55 = w5[:, None] * w5[None, :] / 256.0
    ga, la = [], []

    def put(to, t):
        to.append(t.reshape(-1))
        pad = -t.numel() % 128
        if pad:
            to.append(torch.zeros(pad, dtype=torch.float64, device=DEV))

    for im in images:
        g = im.double()
        for l in range(case["levels"] - 1):
            h, w = g.shape
            h1, w1 = h >> 1, w >> 1
            iy = torch.from_numpy(_map(h, h1).astype(np.int64)).to(DEV)
            ix = torch.from_numpy(_map(w, w1).astype(np.int64)).to(DEV)
            p = _pad(g, 2, 2, capi.CLAMP)
            nxt = torch.zeros((h1, w1), dtype=torch.float64, device=DEV)
            for dy in range(5):
                rows = p[iy + dy]
                for dx in range(5):
                    nxt += w55[dy, dx] * rows[:, ix + dx]
            by = torch.from_numpy(np.maximum(_map(h1, h) - np.float32(0.5), 0).astype(np.float64))
            bx = torch.from_numpy(np.maximum(_map(w1, w) - np.float32(0.5), 0).astype(np.float64))
            by, bx = by.to(DEV), bx.to(DEV)
            yi, xi = by.long(), bx.long()
            fy, fx = (by - yi)[:, None], (bx - xi)[None, :]
            yj, xj = (yi + 1).clamp(max=h1 - 1), (xi + 1).clamp(max=w1 - 1)
            lf = ((1 - fy) * ((1 - fx) * nxt[yi][:, xi] + fx * nxt[yi][:, xj]) +
                  fy * ((1 - fx) * nxt[yj][:, xi] + fx * nxt[yj][:, xj]))
            put(la, g - lf)
            put(ga, nxt)
            g = nxt
    return [torch.cat(ga), torch.cat(la)]


def _exact_train(case, src):
    x, wt, sigma, gy = src
    b = BOUNDARY[case["boundary"]]
    w64 = wt.double().requires_grad_()
    s64 = sigma.double().requires_grad_()
    ys, gxs = [], []
    gw, gs = torch.zeros_like(w64), torch.zeros_like(s64)
    for i in range(case["batch"]):
        xi = x[i].double().requires_grad_()
        y = _bilateral64(_conv64(xi, w64, b), 7, 2.0, s64, b)
        a, bw, bs = torch.autograd.grad(y, (xi, w64, s64), gy[i].double())
        ys.append(y.detach())
        gxs.append(a)
        gw += bw
        gs += bs
    return [torch.stack(ys), torch.stack(gxs), gw.detach(), gs.detach()]


def exact(case, seed):
    kind = case["kind"]
    if case["dtype"] == "u8":
        return None   # bytes and whole numbers
    src = _inputs(case, seed)
    bh = BOUNDARY.get(case.get("boundary"), capi.CLAMP)
    if kind == "train":
        return _exact_train(case, src)
    if kind == "pyramid":
        return _pyramid64(case, src)
    if kind == "rgba":
        w = torch.from_numpy(_gauss(case["k"])).double().to(DEV)
        y = _conv64(src.double().permute(2, 0, 1), w, bh)
        return [y.permute(1, 2, 0).contiguous()]
    x = src.double()
    if kind == "conv":
        return [_conv64(x, torch.from_numpy(_gauss(case["k"])).double().to(DEV), bh)]
    if kind == "separable":
        t = torch.from_numpy(_sep_taps(case["k"])).double().to(DEV)
        return [_conv64(_conv64(x, t[None, :], bh), t[:, None], bh)]
    if kind == "bilateral":
        return [_bilateral64(x, case["k"], case["k"] / 4.0, float(np.float32(0.1)), bh)]
    if kind == "fused":
        w = torch.from_numpy(masks.gaussian_2d(5, 1.0)).double().to(DEV)
        for ch in case["chain"]:
            x = x + 0.25 if ch == "P" else _conv64(x, w, bh)
        return [x]
    if kind == "morph":
        return None   # pixels of the input, chosen by comparisons
    return [x.sum().reshape(1), x.min().reshape(1), x.max().reshape(1), None]
