"""MIN / MAX over whole masks (erode, dilate) against the oracle, bit for bit:
the row-streaming kernel's lane halo, segment ends and partial strips, the
boundary modes, and float windows that hold NaN, infinities and signed zeros
(a NaN tap never replaces the running value; a NaN first tap stays)."""
import numpy as np
import pytest

import oracle_binding as ob
from gpu_util import empty_gpu, to_gpu, to_host
from hipacc_amd import capi, operators as op

pytestmark = pytest.mark.gpu

MODES = [capi.CLAMP, capi.REPEAT, capi.MIRROR, capi.CONSTANT]


def _check(src, k, red, **kw):
    ref = np.zeros_like(src)
    f = src.dtype == np.float32
    ob.local(src, ref, k, k, acc_float=f, reduce=red, **kw)
    dst = empty_gpu(src.shape, src.dtype)
    code = ob.CODES[src.dtype]   # uint16 lives in an int16 tensor
    op.local(to_gpu(src), dst, k, k, acc_float=f, reduce=red, src_dtype=code, dst_dtype=code, **kw)
    got = to_host(dst, src.dtype)
    if f:
        np.testing.assert_array_equal(np.isnan(got), np.isnan(ref))
        keep = ~np.isnan(ref)
        got, ref = got[keep].view(np.uint32), ref[keep].view(np.uint32)
    np.testing.assert_array_equal(got, ref)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("k", [3, 5, 7, 9])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.int16, np.float32])
def test_minmax_vs_oracle(gpu, mode, k, dtype):
    print(f"minmax {np.dtype(dtype).name} k={k} mode={mode}", flush=True)
    for h, w in ((1, 1), (k, 3), (37, 249), (70, 513)):
        if mode == capi.MIRROR and min(h, w) < k // 2:
            continue   # a single reflection does not reach the image
        src = ob.random_image((h, w), dtype, 11 * k + h)
        for red in (capi.MIN, capi.MAX):
            _check(src, k, red, boundary=mode, const_val=3)


@pytest.mark.parametrize("k", [3, 5, 9])
def test_minmax_float_specials(gpu, k):
    rng = np.random.default_rng(k)
    src = rng.choice(np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1.0, -1.0], np.float32),
                     size=(53, 300), p=[.3, .1, .1, .2, .2, .05, .05]).astype(np.float32)
    src[20:40, 100:160] = np.nan
    for red in (capi.MIN, capi.MAX):
        for mode in (capi.CLAMP, capi.CONSTANT):
            _check(src, k, red, boundary=mode, const_val=0.5)


def test_minmax_windows_batches(gpu):
    src = ob.random_image((3, 61, 333), np.uint8, 5)
    _check(src, 5, capi.MIN, boundary=capi.CLAMP)
    one = ob.random_image((61, 333), np.float32, 6)
    for sw in ((3, 2, 320, 55), (8, 0, 256, 61)):
        ref = np.zeros_like(one)
        kw = dict(reduce=capi.MAX, boundary=capi.MIRROR, src_window=sw,
                  dst_window=(1, 0, sw[2], sw[3]))
        ob.local(one, ref, 7, 7, **kw)
        dst = to_gpu(np.zeros_like(one))
        op.local(to_gpu(one), dst, 7, 7, **kw)
        np.testing.assert_array_equal(to_host(dst, np.float32), ref)
