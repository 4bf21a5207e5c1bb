"""Weight gradient of tiles that two FP16 values a number cannot hold: infinities and NaN (which
reach the sums that read them and no other), products and images of very unlike magnitude within
a tile, against the FP64 sums."""
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


def _patches(t):
    return torch.stack([_shift(t, d).flatten(-3) for d in TAPS], dim=-2)


def _exact(img, x, g):
    xd, gd = _patches(x.double()[:, 0]), g.double().reshape(g.shape[0], 1, -1)
    P = torch.cat([_patches(img.double()).flatten(0, 1), torch.ones_like(img[:1], dtype=torch.float64).reshape(1, -1)])
    return (xd * gd).sum(0) @ P.T, (xd * gd).abs().sum(0) @ P.abs().T


def _got(dev, img, x, g):
    from mlpcg_amd import kernels as K
    C = img.shape[0]
    _, gW, gb = K.sm_block_backward(g.to(dev), img.to(dev), x.to(dev), torch.zeros(27, C, 3, 3, 3, device=dev),
                                    torch.zeros(27, device=dev))
    return torch.cat([gW.cpu().double().reshape(27, -1), gb.cpu().double().reshape(27, 1)], dim=1)


# FP32 products and sums: three roundings a term, chains of 64 terms a row, then rows, tiles and waves
def _bound(A):
    return A * (2.0 ** -21 + 128 * 2.0 ** -24)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("where", [(4, 8, 64), (0, 0, 0), (4, 0, 64), (0, 8, 63), (2, 3, 30)])
@pytest.mark.parametrize("which", ["x", "g", "image"])
def test_infinities_reach_what_reads_them(dev, which, where, bad):
    C, B, shape = 2, 3, (5, 9, 65)
    print(f"weight gradient {which} {where} {bad}", flush=True)
    gen = torch.Generator().manual_seed(6)
    img, x, g = torch.rand(C, *shape, generator=gen), torch.randn(B, 1, *shape, generator=gen), torch.randn(B, 1, *shape, generator=gen)
    D, A = _exact(img, x, g)
    inside = lambda d: all(0 <= a + b < n for a, b, n in zip(where, d, shape))
    reads = torch.zeros(27, 27 * C + 1, dtype=torch.bool)
    for k, d in enumerate(TAPS):
        if which == "x" and inside([-v for v in d]):  # the cell that reads it at tap d
            reads[k] = True
        if which == "g" and inside(d):
            reads[k] = True
        if which == "image" and inside([-v for v in d]):
            reads[:, 27 + k] = True
    if which == "image":
        img[(1,) + where] = bad
    else:
        (x if which == "x" else g)[(2, 0) + where] = bad
    got = _got(dev, img, x, g)
    assert torch.isfinite(got[~reads]).all() and torch.all((got - D).abs()[~reads] <= _bound(A)[~reads])
    if which != "image":  # (a cell beyond a tap's reach meets that tap's products of 0 there)
        assert not torch.isfinite(got[reads]).any()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,B,shape", [(1, 1, (9, 17, 130)), (3, 2, (5, 9, 65)), (2, 3, (4, 8, 63)), (1, 1, (7, 1, 70))])
@pytest.mark.parametrize("kind", ["halo", "apart", "outlier", "small rows"])
def test_unlike_magnitudes_within_a_tile(dev, kind, C, B, shape, dtype):
    print(f"weight gradient {kind} {dtype} C={C} B={B} {shape}", flush=True)
    gen = torch.Generator().manual_seed(7)
    img, x, g = torch.rand(C, *shape, generator=gen), torch.randn(B, 1, *shape, generator=gen), torch.randn(B, 1, *shape, generator=gen)
    z = torch.arange(shape[2])
    if kind == "halo":  # x is large where g vanishes, and one cell beyond
        x[..., 20:40] *= 2.0 ** 30
        g[..., 19:41] = 0
    elif kind == "apart":  # x and g are large in turn: no product comes near the bound
        left = z < shape[2] // 2
        x, g = torch.where(left, x * 2.0 ** 30, x), torch.where(left, g, g * 2.0 ** 30)
        x[..., shape[2] // 2 - 2:shape[2] // 2 + 2] = 0
    elif kind == "outlier":  # an image cell dwarfs the others where there is no g
        img[0, 2, 0, 30] = 3e9
        g[..., 28:33] = 0
    elif kind == "small rows":  # and half of the image is far below the rest
        img[..., z > shape[2] // 2] *= 2.0 ** -30
        g[..., :shape[2] // 2 + 2] *= 2.0 ** -40
    img, x, g = (t.to(dtype) for t in (img, x, g))
    got, (D, A) = _got(dev, img, x, g), _exact(img, x, g)
    err = (got - D).abs()
    assert torch.all(err <= _bound(A)), float((err / A).max())
    for c in range(C + 1):
        q = slice(27 * c, 27 * (c + 1)) if c < C else slice(27 * C, 27 * C + 1)
        assert float(err[:, q].norm() / D[:, q].norm()) <= 32 * 2.0 ** -24, c


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,B,d", [(1, 1, 0), (3, 2, 1), (2, 3, 2)])
def test_tiles_that_see_x_in_their_halo_alone(dev, C, B, d, dtype):
    """No centre tap of a 4 x 8 x 64 tile has a product, its neighbours' cells do."""
    shape = (10, 17, 134)
    print(f"weight gradient x in the halo {dtype} C={C} B={B} axis {d}", flush=True)
    gen = torch.Generator().manual_seed(10)
    img, x, g = torch.rand(C, *shape, generator=gen), torch.zeros(B, 1, *shape), torch.randn(B, 1, *shape, generator=gen)
    edge = (4, 8, 64)[d]
    x.narrow(2 + d, edge, 1).copy_(torch.randn(B, 1, *shape, generator=gen).narrow(2 + d, edge, 1))
    img, x, g = (t.to(dtype) for t in (img, x, g))
    got, (D, A) = _got(dev, img, x, g), _exact(img, x, g)
    assert torch.all((got - D).abs() <= _bound(A))
    assert float((got - D).norm() / D.norm()) <= 32 * 2.0 ** -24
