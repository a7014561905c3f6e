"""4-wide pixels through the row stream against the oracle, bit for bit: whole
and partial strips (a strip stores 62, 60 or 58 pixels), masks 3x3 to 7x7,
sums, extremes and division, and the shapes that stay with the tile kernel
(holes in float masks, a constant no pixel holds)."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import to_host
from hipacc_amd import capi, masks, operators as op

pytestmark = pytest.mark.gpu
TORCH = {np.dtype(np.uint8): torch.uint8, np.dtype(np.int32): torch.int32,
         np.dtype(np.float32): torch.float32}


def _check(src, sdt, out, odt, k, **kw):
    h, w = src.shape[:2]
    ref = np.zeros((h, w, 4), out)
    ob.local(src, ref, k, k, src_dtype=sdt, dst_dtype=odt, **kw)
    dst = torch.zeros((h, w, 4), dtype=TORCH[np.dtype(out)], device="cuda")
    op.local(torch.from_numpy(src).cuda(), dst, k, k, src_dtype=sdt, dst_dtype=odt, **kw)
    np.testing.assert_array_equal(to_host(dst, out), ref, err_msg=str(kw))


@pytest.mark.parametrize("mode", [capi.CLAMP, capi.REPEAT, capi.MIRROR, capi.CONSTANT])
@pytest.mark.parametrize("k", [3, 5, 7])
def test_vec4_stream_vs_oracle(gpu, mode, k):
    print(f"vec4 stream k={k} mode={mode}", flush=True)
    hole = np.ones(k * k, np.uint8)
    hole[[0, k]] = 0
    g = masks.gaussian_2d(k, k / 4.0)
    for h, w in ((k, 4), (9, 59), (31, 187)):
        u8 = ob.random_image((h, 4 * w), np.uint8, k + w).reshape(h, w, 4)
        f32 = ob.random_image((h, 4 * w), np.float32, k + h).reshape(h, w, 4)
        u = dict(src=u8, sdt=capi.U8X4, out=np.uint8, odt=capi.U8X4, k=k, boundary=mode)
        f = dict(src=f32, sdt=capi.F32X4, out=np.float32, odt=capi.F32X4, k=k, boundary=mode)
        _check(**u, weights=g, cvt=capi.CVT_ROUND, const_val=7)
        _check(**u, weights=g, cvt=capi.CVT_ROUND, domain=hole, fp_contract=False)
        _check(**u, acc_float=False, post_div=float(k * k), const_val=9)
        _check(**{**u, "out": np.int32, "odt": capi.I32X4}, acc_float=False, const_val=9,
               weights=np.arange(k * k, dtype=np.int32) - 4, domain=hole)
        _check(**f, weights=g, const_val=0.25)
        _check(**f, weights=g, domain=hole)
        for red in (capi.MIN, capi.MAX):
            _check(**u, acc_float=False, reduce=red, const_val=9)
            _check(**f, reduce=red, const_val=0.5)


def test_vec4_constant_outside_the_type(gpu):
    """A constant that no byte holds enters the float sum as given, as in the
    tile kernel."""
    src = torch.from_numpy(ob.random_image((20, 4 * 70), np.uint8, 3).reshape(20, 70, 4)).cuda()
    out = [torch.zeros_like(src) for _ in range(2)]
    for dst, var in zip(out, (capi.VAR_AUTO, capi.VAR_GENERIC)):
        op.prepare_local(src, dst, 5, 5, weights=masks.gaussian_2d(5, 1.0), cvt=capi.CVT_ROUND,
                         boundary=capi.CONSTANT, const_val=300, src_dtype=capi.U8X4,
                         dst_dtype=capi.U8X4).with_variant(var).launch()
    assert torch.equal(out[0], out[1])
