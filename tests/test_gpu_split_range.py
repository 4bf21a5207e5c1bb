"""Blocks on the matrix cores (forward and input gradient) with images, weights, biases and vectors
whose values are further apart than two FP16 parts reach: every result is as good as FP32 sums of
its own terms, infinities stay what they are, and weights below 11 bits count."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
TAPS = list(itertools.product((-1, 0, 1), repeat=3))


def _shift(t, d):
    """t[..., v + d], zero outside."""
    n = t.shape[-3:]
    p = torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1))
    return p[..., 1 + d[0]:1 + d[0] + n[0], 1 + d[1]:1 + d[1] + n[1], 1 + d[2]:1 + d[2] + n[2]]


def _stencils(img, w, b):
    """K [27][grid], FP64, and the sums of its terms' magnitudes."""
    P = torch.stack([_shift(img.double(), d) for d in TAPS], 1).flatten(0, 1).flatten(1)
    W = w.double().reshape(27, -1)
    shape = (27, *img.shape[1:])
    return (W @ P + b.double()[:, None]).view(shape), (W.abs() @ P.abs() + b.double().abs()[:, None]).view(shape)


def _forward(K, x):
    return sum(K[p] * _shift(x.double()[:, 0], d) for p, d in enumerate(TAPS))


def _backward(K, g):
    return sum(_shift(K[p] * g.double()[:, 0], tuple(-a for a in d)) for p, d in enumerate(TAPS))


KINDS = ["outlier", "far outlier", "channels", "channel apart", "rows", "weights", "bias", "huge x", "tiny x", "all small"]


def _inputs(kind, C, B, shape, seed):
    gen = torch.Generator().manual_seed(seed)
    img = torch.rand(C, *shape, generator=gen) + 0.25
    v = torch.randn(B, 1, *shape, generator=gen)
    w = (torch.rand(27, C, 3, 3, 3, generator=gen) - 0.5) * 0.4
    b = (torch.rand(27, generator=gen) - 0.5) * 0.4
    i, j, k = (n // 2 for n in shape)
    if kind == "outlier":
        img[0, i, j, k], b = 1e6, b * 0
    elif kind == "far outlier":
        img[0, i, j, k], img[0, 0, 0, 0], b = 1e12, 3e-7, b * 0
    elif kind == "channels":  # far apart, weights the other way round
        s = torch.tensor([1.0, 2.0 ** -20, 2.0 ** 24][:C])
        img, w = img * s.view(C, 1, 1, 1), w / s.view(1, C, 1, 1, 1)
    elif kind == "channel apart":  # the last channel's products are small, and alone in half of the grid
        img[-1] *= 2.0 ** -24
        if C > 1:
            img[:-1, :, :, k:] = 0
        b = b * 0
    elif kind == "rows":
        img[..., k:] *= 2.0 ** -30
        b = b * 0
    elif kind == "weights":  # small ones alone meet the image on one side of it
        w[:, :, 0] *= 2.0 ** -30
        img[:, :i], img[:, i + 1:], b = 0, 0, b * 0
    elif kind == "bias":  # large on one tap, which most cells' x does not meet
        b = b * 0
        b[14] = 2.0 ** 30
        v[..., :k] = 0
        v[..., k + 1:] = 0
    elif kind == "huge x":
        v = v * 1e30
    elif kind == "tiny x":
        v = v * 1e-30
    elif kind == "all small":
        img, w, b = img * 1e-15, w * 1e-12, b * 1e-27
    return img, v, w, b


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("C,B,shape", [(1, 1, (8, 32, 64)), (3, 2, (9, 29, 66)), (2, 3, (5, 40, 90))])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ranges(dev, dtype, C, B, shape, kind):
    from mlpcg_amd import kernels as K
    print(f"ranges {dtype} C={C} B={B} {shape} {kind}", flush=True)
    img, v, w, b = _inputs(kind, C, B, shape, 3)
    img, v, w, b = img.to(dtype).to(dev), v.to(dtype).to(dev), w.to(dev), b.to(dev)
    k64, mag = _stencils(img, w, b)
    y = K.sm_block_forward(img, v, w, b)[:, 0].double()
    dx = K.sm_block_backward(v, img, torch.ones_like(v), w, b)[0][:, 0].double()
    for got, apply in ((y, _forward), (dx, _backward)):
        ref, m = apply(k64, v), apply(mag, v.abs())
        # K: operands to 2^-23 each, the product of the low parts left out: 2^-21; fewer than 96
        # FP32 roundings in K and the products' sum; FP32's smallest step where x is tiny
        bound = m * (2.0 ** -21 + 96 * 2.0 ** -24) + 27 * 2.0 ** -149
        if dtype == torch.bfloat16:
            bound = bound + ref.abs() * 2.0 ** -8 + 2.0 ** -133
        err = (got - ref).abs()
        assert torch.all(err <= bound), float((err / bound).max())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C", [1, 3])
def test_infinite_values_keep_their_sign(dev, C, dtype):
    """Positive weights and x: an infinite image cell or weight gives infinity, not NaN, where it
    is read, and leaves the other cells alone."""
    from mlpcg_amd import kernels as K
    gen = torch.Generator().manual_seed(4)
    shape = (8, 32, 66)
    img, x = torch.rand(C, *shape, generator=gen) + 0.1, torch.rand(1, 1, *shape, generator=gen) + 0.1
    w, b = torch.rand(27, C, 3, 3, 3, generator=gen) + 0.1, torch.rand(27, generator=gen)
    for what in ("image", "weight", "bias"):
        im, ww, bb = img.clone(), w.clone(), b.clone()
        if what == "image":
            im[C - 1, 3, 7, 63] = float("inf")
        elif what == "weight":
            ww[13, 0, 1, 1, 1] = float("inf")
        else:
            bb[13] = float("inf")
        im, xx, ww, bb = im.to(dtype).to(dev), x.to(dtype).to(dev), ww.to(dev), bb.to(dev)
        y = K.sm_block_forward(im, xx, ww, bb)[0, 0]
        dx = K.sm_block_backward(xx, im, xx, ww, bb)[0][0, 0]
        for got, reach in ((y, 1), (dx, 2)):
            assert not torch.isnan(got).any(), (what, int(torch.isnan(got).sum()))
            near = torch.zeros(shape, dtype=torch.bool)
            near[3 - reach:4 + reach, 7 - reach:8 + reach, 63 - reach:64 + reach] = True
            assert torch.equal(torch.isinf(got).cpu(), near if what == "image" else torch.ones_like(near)), what


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_low_bits_of_the_weights_count(dev, dtype):
    """Weights that differ below 11 bits only, on taps that cancel: the result is their difference."""
    from mlpcg_amd import kernels as K
    shape = (8, 32, 66)
    img, x = torch.ones(1, *shape), torch.ones(1, 1, *shape)
    w, b = torch.zeros(27, 1, 3, 3, 3), torch.zeros(27)
    w[13, 0, 1, 1, 1], w[13, 0, 1, 1, 2] = 1 + 2.0 ** -14, -1.0
    img, x, w, b = img.to(dtype).to(dev), x.to(dtype).to(dev), w.to(dev), b.to(dev)
    y = K.sm_block_forward(img, x, w, b)[0, 0].float()[..., :-1]
    dx = K.sm_block_backward(x, img, x, w, b)[0][0, 0].float()[..., :-1]
    assert torch.all(y == 2.0 ** -14) and torch.all(dx == 2.0 ** -14)
