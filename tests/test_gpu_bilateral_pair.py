"""Bilateral filter and its backward by pixel pairs at sizes the pair kernels
take: several images, widths that end inside a pixel group and inside a wave,
heights that end inside a band and inside a wave's segment, every boundary
mode.  Forward against 64 bits; backward against the 64-bit adjoint with the
adjoint tests' bound (1e-5 of the sum of magnitudes).

The forward bound: sums of n = k*k terms in [0, 1], each with a few float
roundings, are off by less than (n + 10) 2^-24 of the sum of magnitudes, and
so is the quotient; pixels are in [0, 1]."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import to_gpu, to_host
from hipacc_amd import capi, operators as op

pytestmark = pytest.mark.gpu

MODES = [capi.UNDEFINED, capi.CLAMP, capi.REPEAT, capi.MIRROR, capi.CONSTANT]
SHAPE = (5, 517, 1027)
CASES = [(7, m) for m in MODES] + [(5, capi.MIRROR), (5, capi.CONSTANT), (9, capi.CLAMP),
                                    (9, capi.REPEAT)]


@pytest.mark.parametrize("k,mode", CASES + [(11, capi.CLAMP), (13, capi.MIRROR), (15, capi.REPEAT)])
def test_bilateral_pair_forward(gpu, mode, k):
    for shape in (SHAPE, (1, 1501, 2050)):
        print(f"bilateral pair k={k} mode={mode} {shape}", flush=True)
        x = ob.random_image(shape, np.float32, k + mode)
        X = to_gpu(x)
        Y = torch.empty_like(X)
        op.bilateral(X, Y, k, 2.0, 0.3, boundary=mode, const_val=0.5)
        y = to_host(Y, np.float32)
        # whole rows at the top, in the middle and at the bottom, through a
        # crop with the mask's reach (the image's own edge rows at the ends)
        h, r = shape[1], k // 2
        for b in (0, shape[0] - 1):
            for y0, y1 in ((0, 24), (h // 2, h // 2 + 24), (h - 24, h)):
                if mode == capi.REPEAT and (y0 < r or y1 + r > h):
                    crop = np.concatenate([x[b, -r:], x[b, :24 + r]]) if y0 == 0 else \
                        np.concatenate([x[b, y0 - r:], x[b, :r]])
                    lo = r
                else:
                    lo = min(y0, r)
                    crop = x[b, y0 - lo:min(y1 + r, h)]
                f64 = np.zeros(crop.shape, np.float64)
                crop = np.ascontiguousarray(crop)
                ob.bilateral(crop, np.zeros_like(crop), k, 2.0, 0.3, boundary=mode,
                             const_val=0.5, f64_out=f64)
                ref, got = f64[lo:lo + y1 - y0], y[b, y0:y1]
                if mode == capi.UNDEFINED:
                    cut = slice(r if y0 == 0 else 0, -r if y1 == h else None)
                    ref, got = ref[cut, r:-r], got[cut, r:-r]
                assert np.abs(got - ref).max() <= (k * k + 10) * 2.0 ** -24


@pytest.mark.parametrize("k,mode", CASES)
def test_bilateral_pair_backward(gpu, mode, k):
    for shape in (SHAPE,):
        print(f"bilateral pair grad k={k} mode={mode} {shape}", flush=True)
        x = ob.random_image(shape, np.float32, 7 * k + mode)
        g = np.random.default_rng(k).standard_normal(shape).astype(np.float32)
        cval = 0.3 if mode == capi.CONSTANT else 0.0
        dx, ds, dxa, dsa = ob.bilateral_grad(x, g, k, 2.0, 0.1, boundary=mode, const_val=cval,
                                             with_abs=True)
        X, G = to_gpu(x), to_gpu(g)
        Y, D, GX = torch.empty_like(X), torch.empty_like(X), torch.full_like(X, 7.0)
        GS = torch.zeros(1, dtype=torch.float32, device="cuda")
        op.prepare_bilateral_train(X, Y, D, k, 2.0, 0.1, boundary=mode, const_val=cval).launch()
        op.prepare_bilateral_grad(X, Y, D, G, GX, k, 2.0, 0.1, grad_sigma=GS, boundary=mode,
                                  const_val=cval).launch()
        err = np.abs(to_host(GX, np.float32) - dx)
        assert (err <= 1e-5 * dxa + 1e-12).all(), (err / (dxa + 1e-30)).max()
        assert abs(float(GS.item()) - ds) <= 1e-5 * dsa
