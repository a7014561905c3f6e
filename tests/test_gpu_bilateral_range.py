"""Bilateral filter on images whose pixels differ by orders of magnitude, at
sizes the pixel-pair kernels take: hot pixels at the first place of the image
and inside it, a CONSTANT border far from the image, images of one batch in
different units, values up to the ends of the float range, infinities and NaN.
Compared with 64 bits, each pixel by a bound relative to what its own window
may contribute.

Forward bound.  With u = 2^-24 and M = |X(p)| + 8 sigma (a pixel farther from
X(p) than 8 sigma has a weight below 2^-46 of its place in the window, and its
product with the difference is smaller still): each of the n = k*k terms
enters the sums with a few roundings, and a weight s is off by
s (4 |e| + 2) u for its own exponent e (s |e| <= 0.54) and, where the pixels
are scaled before the difference is taken, by another s |t| M u / sigma for
the scaled difference t (s t^2 <= 0.54).  Over the sum of weights, which is at
least the centre's 1, that is less than 2 (n + 10) u M.  The norm has no
division by itself: less than 5 (n + 10) u of it.

The backward is held to the adjoint tests' bound, 1e-5 of the sum of
magnitudes, which is itself a sum over the pixel's window."""
import numpy as np
import pytest
import torch

import oracle_binding as ob
from gpu_util import to_host
from hipacc_amd import capi, operators as op

pytestmark = pytest.mark.gpu

SIGMA, SIGMA_D = 0.1, 2.0
U = 2.0 ** -24
SHAPE = (1, 1501, 2050)
HOT = [1e2, 1e4, 1e6, 1e9, -9999.0, 3.4028234e38]


def _base(shape, seed):
    return torch.rand(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")


def _table(k):
    r = np.arange(k) - k // 2
    d2 = r[:, None] ** 2 + r[None, :] ** 2
    return np.exp(-d2 / (2.0 * SIGMA_D * SIGMA_D)).astype(np.float32)


def _windows(x, k, mode, cval, table=None):
    """(spatial weight, X(p + o)) of every tap, boundary handling applied, in 64 bits."""
    r = k // 2
    h, w = x.shape[-2:]

    def idx(n):
        i = torch.arange(-r, n + r, device="cuda")
        out = (i < 0) | (i >= n)
        if mode == capi.REPEAT:
            i = i % n
        elif mode == capi.MIRROR:
            i = torch.where(i < 0, -i - 1, torch.where(i >= n, 2 * n - 1 - i, i))
        return i.clamp(0, n - 1), out

    (iy, oy), (ix, ox) = idx(h), idx(w)
    p = x.double()[..., iy, :][..., ix]
    if mode == capi.CONSTANT:
        p = p.masked_fill(oy[:, None] | ox[None, :], float(np.float32(cval)))
    table = _table(k) if table is None else table
    for dy in range(k):
        for dx in range(k):
            yield float(table[dy, dx]), p[..., dy:dy + h, dx:dx + w]


def _exact(x, k, sigma, mode, cval, table=None):
    c = x.double()
    num, den = torch.zeros_like(c), torch.zeros_like(c)
    for sp, v in _windows(x, k, mode, cval, table):
        s = torch.exp(-(v - c) ** 2 / (2.0 * float(np.float32(sigma)) ** 2)) * sp
        num += s * v
        den += s
    return num / den, den


def _run(x, k, sigma, mode, cval, train):
    y, n = torch.empty_like(x), torch.empty_like(x)
    if train:
        op.prepare_bilateral_train(x, y, n, k, SIGMA_D, sigma, boundary=mode,
                                   const_val=cval).launch()
    else:
        op.bilateral(x, y, k, SIGMA_D, sigma, boundary=mode, const_val=cval)
    torch.cuda.synchronize()
    return y, n


def _check(x, k, sigma, mode, cval, train, where=None):
    y, n = _run(x, k, sigma, mode, cval, train)
    ey, en = _exact(x, k, sigma, mode, cval)
    where = torch.ones_like(x, dtype=torch.bool) if where is None else where
    t = k * k
    tol = 2 * (t + 10) * U * (x.double().abs() + 8 * sigma)
    bad = ~((y.double() - ey).abs() <= tol) & where
    assert not bad.any(), (int(bad.sum()), ((y.double() - ey).abs() / tol)[where].max().item())
    if train:
        bad = ~((n.double() - en).abs() <= 5 * (t + 10) * U * en) & where
        assert not bad.any(), (int(bad.sum()), ((n.double() - en).abs() / en)[where].max().item())


def _mark(x, value):
    """One marker at the image's first pixel, some inside it, one at its last."""
    h, w = x.shape[-2:]
    for y, c in ((0, 0), (0, w - 1), (h // 3, w // 2), (h // 2, 0), (h // 2, w // 2 + 1),
                 (h - 1, w - 1)):
        x[..., y, c] = value
    return x


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("value", HOT)
@pytest.mark.parametrize("k,mode", [(7, capi.CLAMP), (9, capi.MIRROR), (5, capi.CONSTANT)])
def test_hot_pixels(gpu, k, mode, value, train):
    _check(_mark(_base(SHAPE, 1), value), k, SIGMA, mode, 0.5, train)


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("cval", [-9999.0, 1e6, 1e9, 3.4028234e38])
@pytest.mark.parametrize("k", [5, 7, 13])
def test_far_constant(gpu, k, cval, train):
    _check(_base(SHAPE, 2), k, SIGMA, capi.CONSTANT, cval, train)


@pytest.mark.parametrize("train", [False, True])
def test_images_of_a_batch_in_different_units(gpu, train):
    x = _base((5, 517, 1027), 3)
    x[1] *= 1e6
    x[3] = -1e9
    _check(x, 7, SIGMA, capi.CLAMP, 0.0, train)


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("offset,sigma", [(1000.0, 0.1), (1000.0, 0.01), (0.0, 1e-3),
                                          (0.0, 1e4), (0.0, 1e12), (0.0, 1e-8),
                                          (0.0, 1e-12)])
def test_offset_and_sigma(gpu, offset, sigma, train):
    _check(_base(SHAPE, 4) + offset, 7, sigma, capi.REPEAT, 0.0, train)


@pytest.mark.parametrize("train", [False, True])
def test_both_ends_of_the_float_range(gpu, train):
    """A weight of 0 leaves out even the farthest finite pixel."""
    x = _mark(_base(SHAPE, 5), 3.4028234e38)
    x[..., 200:204, 300] = -3.4028234e38
    x[..., 202, 301] = 3.4028234e38
    x[..., 800, 900] = 2.0e38
    _check(x, 7, SIGMA, capi.CLAMP, 0.0, train)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("train", [False, True])
def test_infinities_and_nan_stay_in_their_windows(gpu, train, value):
    """A window that holds one gives NaN (0 * inf, as in 64 bits), the others
    are not touched."""
    k = 7
    x = _base(SHAPE, 6)
    x[..., 0, 0] = value
    x[..., 700, 1000] = value
    ey, _ = _exact(x, k, SIGMA, capi.CLAMP, 0.0)
    y, _ = _run(x, k, SIGMA, capi.CLAMP, 0.0, train)
    assert torch.equal(torch.isnan(y), torch.isnan(ey))
    assert torch.isnan(ey).any()
    _check(x, k, SIGMA, capi.CLAMP, 0.0, train, ~torch.isnan(ey))


@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("centre", [0.0, 1e-4])
def test_tables_with_a_small_centre(gpu, train, centre):
    """A pixel far from its neighbours that has little part in its own output:
    the image is not negative, so the sums' error is relative to Y."""
    k, sigma = 7, 1e7
    table = _table(k)
    table[k // 2, k // 2] = centre
    x = _mark(_base(SHAPE, 7), 1e6)
    y, n = torch.empty_like(x), torch.empty_like(x)
    if train:
        op.prepare_bilateral_train(x, y, n, k, SIGMA_D, sigma, spatial=table,
                                   boundary=capi.CLAMP).launch()
    else:
        op.bilateral(x, y, k, SIGMA_D, sigma, spatial=table, boundary=capi.CLAMP)
    ey, _ = _exact(x, k, sigma, capi.CLAMP, 0.0, table)
    err = (y.double() - ey).abs() / ey
    assert (err <= 2 * (k * k + 10) * U).all(), err.max().item()


# The backward takes the pair kernel at both sizes; the forward at the larger
# one only (5x5 and 7x7), so the smaller one also has outputs of the tile
# kernel, whose own sums of several pixels near FLT_MAX overflow.
GRAD_SHAPE, BOTH_SHAPE = (3, 620, 1030), (5, 517, 1027)


def _check_grad(x, g, k, mode, cval, images=None):
    y, n, gx = torch.empty_like(x), torch.empty_like(x), torch.full_like(x, 7.0)
    gs = torch.zeros(1, device="cuda")
    op.prepare_bilateral_train(x, y, n, k, SIGMA_D, SIGMA, boundary=mode, const_val=cval).launch()
    op.prepare_bilateral_grad(x, y, n, g, gx, k, SIGMA_D, SIGMA, grad_sigma=gs, boundary=mode,
                              const_val=cval).launch()
    dx, ds, dxa, dsa = ob.bilateral_grad(to_host(x, np.float32), to_host(g, np.float32), k,
                                         SIGMA_D, SIGMA, boundary=mode, const_val=cval,
                                         with_abs=True)
    err = np.abs(to_host(gx, np.float32) - dx)
    for b in range(x.shape[0]) if images is None else images:
        assert (err[b] <= 1e-5 * dxa[b] + 1e-12).all(), (b, (err[b] / (dxa[b] + 1e-30)).max())
    assert abs(float(gs.item()) - ds) <= 1e-5 * dsa


def _gy(shape, seed):
    return torch.randn(shape, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")


@pytest.mark.parametrize("value", HOT)
@pytest.mark.parametrize("k,mode", [(7, capi.CLAMP), (9, capi.MIRROR), (5, capi.CONSTANT)])
def test_hot_pixels_backward(gpu, k, mode, value):
    shape = GRAD_SHAPE if abs(value) < 1e38 else BOTH_SHAPE
    _check_grad(_mark(_base(shape, 11), value), _gy(shape, 12), k, mode, 0.5)


@pytest.mark.parametrize("cval", [-9999.0, 1e6, 1e9, 3.4028234e38])
def test_far_constant_backward(gpu, cval):
    _check_grad(_base(GRAD_SHAPE, 13), _gy(GRAD_SHAPE, 14), 7, capi.CONSTANT, cval)


def test_images_of_a_batch_in_different_units_backward(gpu):
    """The image in other units takes no gradient: its own dX and part of
    dL/dsigma are 0, the other images' are theirs."""
    x, g = _base(GRAD_SHAPE, 15), _gy(GRAD_SHAPE, 16)
    x[1] *= 1e6
    g[1] = 0.0
    _check_grad(x, g, 7, capi.REPEAT, 0.0)


def test_backward_takes_outputs_rounded_by_any_kernel(gpu):
    """A flat image of large values with Y one last place off (a quotient of
    sums may be): every difference is 0, so dX is the weights' own adjoint and
    dL/dsigma is 0."""
    k = 7
    x, g = torch.full(GRAD_SHAPE, 1e6, device="cuda"), _gy(GRAD_SHAPE, 18)
    y, n, gx = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    gs = torch.zeros(1, device="cuda")
    op.prepare_bilateral_train(x, y, n, k, SIGMA_D, SIGMA, boundary=capi.CLAMP).launch()
    y = torch.nextafter(x, 2 * x)
    op.prepare_bilateral_grad(x, y, n, g, gx, k, SIGMA_D, SIGMA, grad_sigma=gs,
                              boundary=capi.CLAMP).launch()
    dx, _, dxa, _ = ob.bilateral_grad(to_host(x, np.float32), to_host(g, np.float32), k, SIGMA_D,
                                      SIGMA, boundary=capi.CLAMP, with_abs=True)
    err = np.abs(to_host(gx, np.float32) - dx)
    assert (err <= 1e-5 * dxa + 1e-12).all(), (err / dxa).max()
    assert float(gs.item()) == 0.0
