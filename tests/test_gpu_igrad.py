"""Input gradient of a block on the matrix cores (igrad.hpp) against the FP64 scatter at the edges
of its tiles (4 planes, 4, 8 or 16 rows, 64 z cells), for batches that share K in pairs or need
several passes of the workspace, and with values far from FP16's range."""
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


def _reference(img, g, w, b):
    """dx and the sum of the magnitudes of its terms, FP64."""
    P = torch.cat([_shift(img, d)[:, None] for d in TAPS], 1).flatten(0, 1)  # [27 C][grid], channel major
    W = w.double().reshape(27, -1)
    dx, mag = torch.zeros_like(g), torch.zeros_like(g)
    for p, d in enumerate(TAPS):
        K = (W[p] @ P.flatten(1)).reshape(P.shape[1:]) + b.double()[p]
        A = (W[p].abs() @ P.abs().flatten(1)).reshape(P.shape[1:]) + b.double()[p].abs()
        back = tuple(-v for v in d)
        dx += _shift(K * g, back)
        mag += _shift(A * g.abs(), back)
    return dx, mag


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("C,B,shape,kind", [(1, 1, (4, 16, 256), "random"), (3, 3, (5, 17, 195), "random"), (2, 2, (33, 21, 31), "random"),
                                            (1, 2, (1, 129, 128), "random"), (1, 1, (129, 1, 129), "random"), (1, 5, (130, 128, 1), "random"),
                                            (3, 1, (9, 40, 65), "flags"), (1, 2, (12, 23, 127), "far"), (1, 2, (128, 128, 128), "random"),
                                            (3, 1, (64, 132, 130), "random"), (1, 1, (131, 61, 193), "flags")])
def test_input_gradient(dev, dtype, C, B, shape, kind):
    from mlpcg_amd import kernels as K
    print(f"input gradient {dtype} C={C} B={B} {shape} {kind}", flush=True)
    gen = torch.Generator().manual_seed(5)
    img = torch.rand(C, *shape, generator=gen)
    if kind == "flags":
        img = (img > 0.5).float()
    g = torch.randn(B, 1, *shape, generator=gen)
    w = (torch.rand(27, C, 3, 3, 3, generator=gen) - 0.5) * 0.4
    b = (torch.rand(27, generator=gen) - 0.5) * 0.4
    if kind == "far":
        img, b, g = img * 2.0 ** 40, b * 2.0 ** 41, g * 2.0 ** -70
    img, g, w, b = (t.to(dev) for t in (img.to(dtype), g.to(dtype), w, b))
    dx, _, _ = K.sm_block_backward(g, img, torch.randn_like(g), w, b)
    ref, mag = _reference(img.double(), g.double()[:, 0], w, b)
    err = (dx[:, 0].double() - ref).abs()
    if dtype == torch.float32:
        # K: operands to 2^-23 each and the product of the low parts left out, 2^-21; fewer than
        # 32 FP32 roundings in K and 32 in the sum of the 27 products
        bound = mag * (2.0 ** -21 + 64 * 2.0 ** -24)
        norm = 32 * 2.0 ** -24
    else:
        # room for weights of 11 bits, 2^-12, FP32 sums, the result rounded to BF16
        bound = mag * (2.0 ** -12 + 64 * 2.0 ** -24) + ref.abs() * 2.0 ** -8
        norm = 2.0 ** -8
    tiny = float(mag.max()) * 2.0 ** -40
    assert torch.all(err <= bound + tiny), float((err / (bound + tiny)).max())
    assert float(err.norm() / ref.norm()) <= norm


@pytest.mark.parametrize("where", [(0, 0, 0), (3, 7, 63), (4, 8, 64), (8, 39, 64), (5, 20, 31)])
def test_infinities_stay_local(dev, where):
    """An infinite g reaches the 27 cells around it, an infinite image value the 125, and no
    other lane, row, plane or tile."""
    from mlpcg_amd import kernels as K
    gen = torch.Generator().manual_seed(2)
    shape = (9, 40, 65)
    img, g = torch.rand(2, *shape, generator=gen).to(dev), torch.randn(1, 1, *shape, generator=gen).to(dev)
    w, b = torch.randn(27, 2, 3, 3, 3, generator=gen).to(dev), torch.randn(27, generator=gen).to(dev)
    x = torch.randn_like(g)
    dx0 = K.sm_block_backward(g, img, x, w, b)[0][0, 0]
    dist = torch.zeros(shape, device=dev)
    for a, (n, c) in enumerate(zip(shape, where)):
        dist = torch.maximum(dist, (torch.arange(n, device=dev) - c).abs().float().reshape([-1 if k == a else 1 for k in range(3)]))
    bad = g.clone()
    bad[(0, 0) + where] = float("inf")
    dx = K.sm_block_backward(bad, img, x, w, b)[0][0, 0]
    assert torch.equal(torch.isfinite(dx), dist > 1) and torch.allclose(dx[dist > 1], dx0[dist > 1], rtol=1e-5, atol=1e-5)
    bad = img.clone()
    bad[(1,) + where] = float("inf")
    dx = K.sm_block_backward(g, bad, x, w, b)[0][0, 0]
    assert torch.isfinite(dx[dist > 2]).all() and not torch.isfinite(dx[dist <= 1]).any()
    assert torch.allclose(dx[dist > 2], dx0[dist > 2], rtol=1e-5, atol=1e-4)
