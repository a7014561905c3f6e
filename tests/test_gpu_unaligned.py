"""Rows at any alignment: images cut out of wider buffers (first column and
pitch odd, so that neither rows nor their outputs are word-aligned) through
the kernels that read and write whole words, against the oracle, with a check
that nothing outside the output image was written."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import empty_gpu, to_gpu, to_host
from hipacc_amd import capi, masks, operators as op

pytestmark = pytest.mark.gpu

MODES = [capi.UNDEFINED, capi.CLAMP, capi.REPEAT, capi.MIRROR, capi.CONSTANT]
W, H = 1003, 37   # several strips of 248 columns and a partial one; partial row chunks
DT = {np.dtype(np.uint8): torch.uint8, np.dtype(np.float32): torch.float32,
      np.dtype(np.int16): torch.int16, np.dtype(np.uint32): torch.int32}
FILL = 77


def _cut(a, x0, pad):
    """Device image with `x0` columns before and `pad` after each row."""
    h, w = a.shape
    buf = torch.zeros((h, x0 + w + pad), dtype=DT[a.dtype], device="cuda")
    buf[:, x0:x0 + w] = to_gpu(a)
    return buf[:, x0:x0 + w]


def _run(fn, src, out, r, mode, ref, x0=1, **kw):
    buf = empty_gpu((H + 2, W + 6), out, fill=FILL)
    dst = buf[1:H + 1, x0:x0 + W]
    fn(_cut(src, x0, 2), dst, **kw)
    got = to_host(dst, out)
    if mode == capi.UNDEFINED:   # reads beside the image, in the wider buffer
        got, ref = got[r:-r, r:-r], ref[r:-r, r:-r]
    np.testing.assert_array_equal(got, ref)
    buf[1:H + 1, x0:x0 + W] = FILL
    assert bool((buf == FILL).all()), "a pixel outside the output image was written"


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("k", [3, 5, 7, 9, 13])
def test_local_unaligned(gpu, mode, k):
    print(f"unaligned local k={k} mode={mode}", flush=True)
    r, g = k // 2, masks.gaussian_2d(k, k / 4)
    for x0 in (1, 4):   # odd columns; aligned columns with an odd pitch
        src = ob.random_image((H, W), np.float32, k + x0)
        ref = np.zeros_like(src)
        kw = dict(mask_w=k, mask_h=k, weights=g, boundary=mode, const_val=0.5)
        ob.local(src, ref, **kw)
        _run(op.local, src, np.float32, r, mode, ref, x0, **kw)
        u8 = ob.random_image((H, W), np.uint8, k + x0)
        ref = np.zeros_like(u8)
        kw = dict(mask_w=k, mask_h=k, weights=g, boundary=mode, const_val=9, cvt=capi.CVT_ROUND)
        ob.local(u8, ref, **kw)
        _run(op.local, u8, np.uint8, r, mode, ref, x0, **kw)
        if k <= 7:
            w = np.arange(k * k, dtype=np.int32) - k
            ref = np.zeros(u8.shape, np.int16)
            kw = dict(mask_w=k, mask_h=k, weights=w, acc_float=False, boundary=mode, const_val=9)
            ob.local(u8, ref, **kw)
            _run(op.local, u8, np.int16, r, mode, ref, x0, **kw)
            ref = np.zeros_like(u8)
            kw = dict(mask_w=k, mask_h=k, acc_float=False, reduce=capi.MIN, boundary=mode,
                      const_val=9)
            ob.local(u8, ref, **kw)
            _run(op.local, u8, np.uint8, r, mode, ref, x0, **kw)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("k", [3, 5, 7, 9, 13])
def test_separable_unaligned(gpu, mode, k):
    print(f"unaligned separable k={k} mode={mode}", flush=True)
    r, g = k // 2, masks.gaussian_1d(k, k / 4)
    src, u8 = ob.random_image((H, W), np.float32, k), ob.random_image((H, W), np.uint8, k)
    ref = np.zeros_like(src)
    ob.separable(src, ref, g, g, boundary=mode, const_val=0.5)
    _run(op.separable, src, np.float32, r, mode, ref, row=g, col=g, boundary=mode, const_val=0.5)
    ref = np.zeros_like(u8)
    kw = dict(boundary=mode, const_val=9, cvt=capi.CVT_ROUND)
    ob.separable(u8, ref, g, g, **kw)
    _run(op.separable, u8, np.uint8, r, mode, ref, row=g, col=g, **kw)
    if k <= 7:
        ones = np.ones(k, np.int32)
        for out, code in ((np.int16, capi.I16), (np.uint32, capi.U32)):
            ref = np.zeros(u8.shape, out)
            kw = dict(acc_float=False, boundary=mode, const_val=9)
            ob.separable(u8, ref, ones, ones, **kw)
            _run(op.separable, u8, out, r, mode, ref, row=ones, col=ones, dst_dtype=code, **kw)


@pytest.mark.parametrize("mode", MODES)
def test_bilateral_unaligned(gpu, mode):
    """The aligned copy of the image gives the same bits."""
    for dtype, sr in ((np.float32, 0.2), (np.uint8, 25.0)):
        src = ob.random_image((H, W), dtype, 5)
        cvt = capi.CVT_ROUND if dtype == np.uint8 else capi.CVT_TRUNC
        pitched = to_gpu(src, pitch=1024)
        ref = torch.zeros_like(pitched)
        op.bilateral(pitched, ref, 7, 2.0, sr, boundary=mode, const_val=0.5, cvt=cvt)
        _run(op.bilateral, src, dtype, 3, mode, to_host(ref, dtype), ksize=7, sigma_d=2.0,
             sigma_r=sr, boundary=mode, const_val=0.5, cvt=cvt)


@pytest.mark.parametrize("dtype", [np.uint8, np.float32])
def test_global_operators_unaligned(gpu, dtype):
    """Reductions and histograms over rows back to back from any first byte and
    over pitched rows of every tail length.  Small integers: float sums exact."""
    f = dtype == np.float32
    for h, w in ((1, 1), (3, 5), (5, 17), (37, 1003), (64, 255)):
        src = np.random.default_rng(w).integers(0, 200, (h, w)).astype(dtype)
        flat = torch.zeros(h * w + 3, dtype=DT[np.dtype(dtype)], device="cuda")
        for off in (0, 1, 3):
            flat[off:off + h * w] = to_gpu(src).flatten()
            for img in (flat[off:off + h * w].view(h, w), _cut(src, off, 2)):
                for red, ref in ((capi.SUM, src.astype(np.float64).sum()), (capi.MIN, src.min()),
                                 (capi.MAX, src.max())):
                    res = torch.zeros(1, dtype=torch.float32 if f else torch.int32, device="cuda")
                    op.reduce(img, red, res)
                    assert float(res.item()) == float(ref)
                bins = torch.zeros(256, dtype=torch.int32, device="cuda")
                op.histogram(img, 256, bins)
                np.testing.assert_array_equal(to_host(bins, np.int32),
                                              np.bincount(src.astype(np.int64).ravel(),
                                                          minlength=256))


@pytest.mark.parametrize("dt", [np.uint8, np.float32])
@pytest.mark.parametrize("nbins", [256, 4096])
def test_histogram_routes(gpu, dt, nbins):
    """Contiguous windows around the sizes where the share of a block changes,
    and pitched rows, aligned or not, on either side of the widths that are
    read as vectors."""
    eb = np.dtype(dt).itemsize
    shapes = [(1, n // eb) for n in (4095, 4100, 64 * 4096 + 4, 192 * 16384 - 4, 192 * 65536 + 4)]
    shapes += [(h, w) for w in (15, 1199, 1200, 2047, 2048, 2049) for h in (3, 700)]
    for h, w in shapes:
        a = ob.random_image((h, w), dt, w + nbins)
        scale = float(nbins) if dt == np.float32 else 1.0
        ref = ob.histogram(a, nbins, scale)
        for x0, pad in ((0, 0), (1, 0), (1, 2), (16, 16 + -w % 16)):
            bins = torch.full((nbins,), -1, dtype=torch.int32, device="cuda")
            if pad:
                src = _cut(a, x0, pad)
            else:   # rows back to back, the first one x0 pixels into the buffer
                flat = torch.zeros(h * w + x0, dtype=DT[a.dtype], device="cuda")
                flat[x0:] = to_gpu(a).reshape(-1)
                src = flat[x0:].view(h, w)
            op.histogram(src, nbins, bins, scale=scale)
            np.testing.assert_array_equal(to_host(bins, np.uint32), ref, err_msg=f"{h}x{w} {x0} {pad}")
