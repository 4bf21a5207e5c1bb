"""Weight gradient of grids whose workgroups take several tiles of unlike magnitude: empty tiles,
tiles whose x and g are large in turn, right-hand sides of zeros, channels of unlike scale,
against the FP64 sums."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


def _shift(t, d):
    """t[..., v + d], zero outside."""
    n = t.shape[-3:]
    p = torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1))
    return p[..., 1 + d[0]:1 + d[0] + n[0], 1 + d[1]:1 + d[1] + n[1], 1 + d[2]:1 + d[2] + n[2]]


def _patches(t):
    """(..., 27, V) of (..., n1, n2, n3)."""
    return torch.stack([_shift(t, d).flatten(-3) for d in itertools.product((-1, 0, 1), repeat=3)], dim=-2)


def _exact(img, x, g):
    """D [27][27 C + 1] and the sums of the magnitudes of its terms, FP64."""
    xd, gd = _patches(x.double()[:, 0]), g.double().reshape(g.shape[0], 1, -1)
    P = torch.cat([_patches(img.double()).flatten(0, 1), torch.ones_like(img[:1], dtype=torch.float64).reshape(1, -1)])
    return (xd * gd).sum(0) @ P.T, (xd * gd).abs().sum(0) @ P.abs().T


def _got(dev, img, x, g):
    from mlpcg_amd import kernels as K
    C = img.shape[0]
    _, gW, gb = K.sm_block_backward(g, img, x, torch.zeros(27, C, 3, 3, 3, device=dev), torch.zeros(27, device=dev))
    return torch.cat([gW.double().reshape(27, -1), gb.double().reshape(27, 1)], dim=1)


# (130, 128, 1): 528 tiles in 65 workgroups; (260, 40, 3): 325 tiles in 122
@pytest.mark.parametrize("kind", ["plain", "empty", "in turn", "batch", "channels", "channels in turn"])
@pytest.mark.parametrize("shape", [(130, 128, 1), (260, 40, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_tiles_of_unlike_magnitude(dev, dtype, shape, kind):
    print(f"weight gradient {dtype} {shape} {kind}", flush=True)
    C, B = (3, 1) if kind.startswith("channels") else (1, 3)
    gen = torch.Generator().manual_seed(3)
    img = torch.rand(C, *shape, generator=gen)
    x = torch.randn(B, 1, *shape, generator=gen)
    g = torch.randn(B, 1, *shape, generator=gen)
    # tiles in turn by planes of 4 (a workgroup meets both sorts, whichever way it walks); where
    # the tiles' magnitudes differ, zeros keep them from being each other's halo
    border = torch.isin(torch.arange(shape[0]) % 4, torch.tensor([0, 3])).view(-1, 1, 1)
    odd = ((torch.arange(shape[0]) // 4) % 2 == 1).view(-1, 1, 1)
    third = ((torch.arange(shape[0]) // 4) % 3 == 1).view(-1, 1, 1)
    if kind == "empty":
        g, x = g * 1e-9, torch.where(third, x * 1e-3, torch.zeros(()))
        g = torch.where(third, g, torch.zeros(()))
    elif kind == "in turn":
        x, g = torch.where(odd, x * 2.0 ** 20, x * 2.0 ** -20), torch.where(odd, g * 2.0 ** -20, g * 2.0 ** 20)
        x = torch.where(border, torch.zeros(()), x)
    elif kind == "batch":  # an empty first pair; then a pair of unlike sizes
        x[:2] = 0
        g = g * 1e-10
    elif kind == "channels":
        img *= torch.tensor([1.0, 2.0 ** -24, 2.0 ** 24]).view(3, 1, 1, 1)
    elif kind == "channels in turn":
        img = torch.where(border, torch.zeros(()), torch.where(odd, img * 2.0 ** 18, img * 2.0 ** -18))
        g = torch.where(odd, g * 2.0 ** -18, g * 2.0 ** 18)
    img, x, g = (t.to(dtype).to(dev) for t in (img, x, g))
    got, (D, A) = _got(dev, img, x, g), _exact(img, x, g)
    # products: two FP16 values hold G and P to 2^-23 each, G is rounded once per right-hand side,
    # the product of the low parts is left out: 2^-21; sums: fewer than 128 FP32 roundings in a row
    err = (got - D).abs()
    assert torch.all(err <= A * (2.0 ** -21 + 128 * 2.0 ** -24)), float((err / A).max())
    # terms of both signs: the roundings add up at random; by channel
    for c in range(C + 1):
        q = slice(27 * c, 27 * (c + 1)) if c < C else slice(27 * C, 27 * C + 1)
        assert float(err[:, q].norm() / D[:, q].norm()) <= 16 * 2.0 ** -24, c


def test_right_hand_sides_of_unlike_magnitude(dev):
    """Two right-hand sides, x of one and g of the other large: both products matter."""
    gen = torch.Generator().manual_seed(4)
    shape = (9, 17, 70)
    img, x, g = torch.rand(1, *shape, generator=gen), torch.randn(2, 1, *shape, generator=gen), torch.randn(2, 1, *shape, generator=gen)
    for k in (0, 1):
        x[k] *= 2.0 ** (30 if k else -30)
        g[k] *= 2.0 ** (-30 if k else 30)
    img, x, g = (t.to(dev) for t in (img, x, g))
    got, (D, A) = _got(dev, img, x, g), _exact(img, x, g)
    assert torch.all((got - D).abs() <= A * (2.0 ** -21 + 128 * 2.0 ** -24))
    assert float((got - D).norm() / D.norm()) <= 16 * 2.0 ** -24
