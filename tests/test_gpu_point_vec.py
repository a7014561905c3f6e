"""Point operators in whole vectors: every tail length of a row, rows back to
back and pitched, and the integer MAGNITUDE without divisions (quotients by
any norm and square roots next to integers), bit for bit against the oracle."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import empty_gpu, to_gpu, to_host
from hipacc_amd import capi, operators as op

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tin,tout", [(np.uint8, np.uint8), (np.int16, np.uint8),
                                      (np.uint8, np.float32), (np.float32, np.float32),
                                      (np.float32, np.uint8), (np.int32, np.int16)])
def test_point_tails(gpu, tin, tout):
    kw = dict(src_dtype=ob.CODES[np.dtype(tin)], dst_dtype=ob.CODES[np.dtype(tout)])
    for w in list(range(1, 18)) + [255, 4097]:
        for h, pitch in ((1, 0), (3, 0), (3, w + 5)):
            a, b = (ob.random_image((h, w), tin, s + w) for s in (1, 2))
            for code, alpha in ((capi.POINT_AFFINE, 0.5), (capi.POINT_SUB, 1.0)):
                two = code == capi.POINT_SUB
                ref = np.zeros((h, w), tout)
                ob.point(code, a, ref, b if two else None, alpha=alpha, beta=1.0)
                buf = empty_gpu((h + 1, pitch or w), tout, fill=77)
                dst = buf[:h, :w]
                op.point(code, to_gpu(a, pitch), dst, to_gpu(b, pitch) if two else None,
                         alpha=alpha, beta=1.0, **kw)
                np.testing.assert_array_equal(to_host(dst, tout), ref)
                dst[:] = 77
                assert bool((buf == 77).all())


@pytest.mark.parametrize("norm", [0, 1, 2, 3, 4, 7, 181, 255, 1000, 40000, -5])
def test_magnitude_without_division(gpu, norm):
    """All 16-bit values against others that make the sum of squares a square,
    one more and one less; overflowing sums wrap."""
    a = np.arange(-32768, 32768, dtype=np.int16).reshape(256, 256)
    others = [np.zeros_like(a), a, np.full_like(a, 4), np.full_like(a, -1),
              np.full_like(a, -32768), ob.random_image(a.shape, np.int16, norm & 255)]
    for tin in (np.int16, np.uint16):
        code = ob.CODES[np.dtype(tin)]
        for b in others:
            for tout, cvt in ((np.uint8, capi.CVT_TRUNC), (np.uint8, capi.CVT_ROUND),
                              (np.int16, capi.CVT_TRUNC)):
                ref = np.zeros(a.shape, tout)
                ob.point(capi.POINT_MAGNITUDE, a.view(tin), ref, b.view(tin), alpha=float(norm),
                         cvt=cvt)
                dst = empty_gpu(a.shape, tout)
                op.point(capi.POINT_MAGNITUDE, to_gpu(a.view(tin)), dst, to_gpu(b.view(tin)),
                         alpha=float(norm), cvt=cvt, src_dtype=code,
                         dst_dtype=ob.CODES[np.dtype(tout)])
                np.testing.assert_array_equal(to_host(dst, tout), ref)


def test_absdiff_of_int32_wraps(gpu):
    """Differences beyond the int32 range wrap, and the magnitude of INT_MIN is
    INT_MIN, in point calls and in fused chains, also where the result becomes
    float."""
    vals = np.array([-2**31, 2**31 - 1, 0, 1, -1, 5], np.int32)
    a, b = (np.ascontiguousarray(v) for v in np.meshgrid(np.tile(vals, 11), vals))
    with np.errstate(over="ignore"):
        ref = np.abs(a - b).astype(np.float32)
    A, B = to_gpu(a), to_gpu(b)
    for run in (lambda o: op.point(capi.POINT_ABSDIFF, A, o, B),
                lambda o: op.fused(A, o, [dict(kind="point", dtype=capi.F32,
                                               op=capi.POINT_ABSDIFF, in1=B)])):
        out = torch.empty(a.shape, dtype=torch.float32, device="cuda")
        run(out)
        np.testing.assert_array_equal(to_host(out, np.float32), ref)


@pytest.mark.parametrize("tin,tout", [(np.uint8, np.uint8), (np.int16, np.float32)])
def test_point_blocks_of_several_rows(gpu, tin, tout):
    """Rows of fewer than 256 vectors share a block: widths around 2^k vectors,
    heights around the block's rows, tails of every kind of length."""
    kw = dict(src_dtype=ob.CODES[np.dtype(tin)], dst_dtype=ob.CODES[np.dtype(tout)])
    n = 16 // max(np.dtype(tin).itemsize, np.dtype(tout).itemsize)
    for vecs in (1, 2, 8, 45, 128, 256):
        for w in (n * vecs - 1, n * vecs, n * vecs + 1, n * vecs + n // 2):
            rows = 256 >> min(8, int(np.ceil(np.log2(max(1, -(-w // n))))))
            for h in (1, rows, 2 * rows + 1):
                a, b = (ob.random_image((h, w), tin, s + w) for s in (3, 4))
                ref = np.zeros((h, w), tout)
                ob.point(capi.POINT_SUB, a, ref, b)
                buf = empty_gpu((h + 1, w + 3), tout, fill=77)
                op.point(capi.POINT_SUB, to_gpu(a, w + 1), buf[:h, 1:w + 1], to_gpu(b), **kw)
                np.testing.assert_array_equal(to_host(buf[:h, 1:w + 1], tout), ref)
                buf[:h, 1:w + 1] = 77
                assert bool((buf == 77).all())
