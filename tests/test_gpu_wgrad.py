"""Weight gradient on the matrix cores (FP32, and BF16 / FP16 off the 64-cell segments) against
the FP64 sums at the edges of its 4 x 8 x 64 tiles, with odd batches and with values far from
FP16's range."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu

TAPS = list(itertools.product((-1, 0, 1), repeat=3))


def _patches(t):
    """(..., 27, V) of (..., n1, n2, n3): the neighbours, zero outside."""
    n = t.shape[-3:]
    p = torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1))
    return torch.stack([p[..., 1 + d[0]:1 + d[0] + n[0], 1 + d[1]:1 + d[1] + n[1], 1 + d[2]:1 + d[2] + n[2]].flatten(-3)
                        for d in TAPS], dim=-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("C,B,shape,kind", [(1, 1, (1, 1, 1), "random"), (3, 3, (5, 9, 65), "random"), (1, 2, (4, 8, 64), "random"),
                                            (2, 1, (3, 17, 130), "random"), (1, 5, (7, 6, 33), "random"), (3, 1, (8, 16, 63), "flags"),
                                            (1, 2, (12, 9, 70), "far"), (1, 1, (48, 70, 66), "random")])
def test_weight_gradient(dev, dtype, C, B, shape, kind):
    from mlpcg_amd import kernels as K
    print(f"weight gradient {dtype} C={C} B={B} {shape} {kind}", flush=True)
    gen = torch.Generator().manual_seed(9)
    img = torch.rand(C, *shape, generator=gen)
    x = torch.randn(B, 1, *shape, generator=gen)
    g = torch.randn(B, 1, *shape, generator=gen)
    if kind == "flags":
        img = (img > 0.5).float()
    if kind == "far":  # factors differ by tile; FP16 data stays in its own range
        x[..., :20] *= 2.0 ** 9
        g = g * 2.0 ** (-13 if dtype == torch.float16 else -70)
        img = img * 2.0 ** (9 if dtype == torch.float16 else 40)
    img, x, g = (t.to(dtype) for t in (img, x, g))
    w, b = torch.zeros(27, C, 3, 3, 3), torch.zeros(27)
    _, gW, gb = K.sm_block_backward(g.to(dev), img.to(dev), x.to(dev), w.to(dev), b.to(dev))
    xd, gd = _patches(x.double()[:, 0]), g.double().reshape(B, 1, -1)
    P = torch.cat([_patches(img.double()).flatten(0, 1), torch.ones(1, img[0].numel(), dtype=torch.float64)])
    G = (xd * gd).sum(0)
    D = G @ P.T
    got = torch.cat([gW.cpu().double().reshape(27, -1), gb.cpu().double().reshape(27, 1)], dim=1)
    # products: two FP16 values hold G and P to 2^-23 each, G is rounded once in FP32, and the
    # product of the low parts is left out: 2^-21; sums: fewer than 96 FP32 roundings in a row
    A = (xd * gd).abs().sum(0) @ P.abs().T
    floor = 2.0 ** -30 * float((xd.abs().amax() * gd.abs().amax()) * P.shape[1])
    bound = A * (2.0 ** -21 + 96 * 2.0 ** -24) + floor * P.abs().amax(1)
    assert torch.all((got - D).abs() <= bound), float(((got - D).abs() / bound).max())
    # sums of values of both signs: the roundings add up at random (sqrt(96) half-ulps)
    if kind != "far" and D.numel() and img[0].numel() > 1:
        assert float((got - D).norm() / D.norm()) <= 10 * 2.0 ** -24


def test_weight_gradient_keeps_infinities(dev):
    """An infinite x or g makes every entry it enters non-finite and does not disturb the scale
    of the others: an infinite image cell leaves the bias gradient and the other channel alone."""
    from mlpcg_amd import kernels as K
    gen = torch.Generator().manual_seed(1)
    img = torch.rand(2, 9, 10, 70, generator=gen)
    x, g = torch.randn(1, 1, 9, 10, 70, generator=gen), torch.randn(1, 1, 9, 10, 70, generator=gen)
    w, b = torch.zeros(27, 2, 3, 3, 3, device=dev), torch.zeros(27, device=dev)
    _, gW0, gb0 = K.sm_block_backward(g.to(dev), img.to(dev), x.to(dev), w, b)
    bad = img.clone()
    bad[1, 4, 5, 30] = float("inf")
    _, gW, gb = K.sm_block_backward(g.to(dev), bad.to(dev), x.to(dev), w, b)
    assert torch.allclose(gb, gb0, rtol=1e-5, atol=1e-5) and torch.allclose(gW[:, 0], gW0[:, 0], rtol=1e-5, atol=1e-4)
    assert not torch.isfinite(gW[:, 1]).any()
    bad = x.clone()
    bad[0, 0, 4, 5, 30] = float("inf")
    _, gW, gb = K.sm_block_backward(g.to(dev), img.to(dev), bad.to(dev), w, b)
    assert not torch.isfinite(gb).any() and not torch.isfinite(gW).any()
