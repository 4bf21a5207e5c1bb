"""Mean patch from the sums over the grid's disjoint parts: infinities and large values at the
faces reach the offsets that include them and no other; grids of one and two cells an axis."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
OFFSETS = list(itertools.product((-1, 0, 1), repeat=3))


def _patch(img):
    """ybar [C][27] in FP64: the mean over v of img[v + e], zero outside."""
    out = torch.zeros(img.shape[0], 27, dtype=torch.float64)
    for k, d in enumerate(OFFSETS):
        s = tuple(slice(max(a, 0), n + min(a, 0)) for a, n in zip(d, img.shape[1:]))
        out[:, k] = img.double()[(slice(None),) + s].flatten(1).sum(1)
    return out / img[0].numel()


SHAPES = [(1, 1, 1), (2, 1, 3), (1, 5, 2), (2, 2, 2), (3, 2, 8), (5, 6, 12), (33, 17, 65), (24, 40, 100)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
def test_every_offset(dev, shape, dtype):
    from mlpcg_amd import kernels as K
    print(f"mean patch {dtype} {shape}", flush=True)
    gen = torch.Generator().manual_seed(8)
    for C in (1, 3):
        img = (torch.rand(C, *shape, generator=gen, dtype=torch.float64) - 0.3).to(dtype)
        acc = torch.float64 if dtype == torch.float64 else torch.float32
        w, b = torch.randn(1, C, 3, 3, 3, generator=gen, dtype=acc), torch.randn(1, generator=gen, dtype=acc)
        z, ybar = K.sm_linear(img.to(dev), w.to(dev), b.to(dev))
        ref = _patch(img)
        # FP64 sums, rounded once to the accumulation type
        eps = 2.0 ** -24 if acc == torch.float32 else 2.0 ** -45
        assert torch.all((ybar.cpu().double().view(C, 27) - ref).abs() <= eps * ref.abs() + 2.0 ** -45)
        zr = (w.double().view(-1) * ybar.cpu().double().view(-1)).sum() + b.double()
        assert abs(float(z.cpu().double() - zr)) <= 4 * eps * (1 + abs(float(zr)))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 1e36])
@pytest.mark.parametrize("shape", [(3, 2, 8), (5, 6, 12), (33, 17, 65), (24, 40, 100)])
def test_faces_reach_their_offsets_alone(dev, shape, value, dtype):
    from mlpcg_amd import kernels as K
    print(f"mean patch {dtype} {shape} {value}", flush=True)
    gen = torch.Generator().manual_seed(9)
    base = torch.rand(2, *shape, generator=gen).to(dtype)
    n1, n2, n3 = shape
    w, b = torch.zeros(1, 2, 3, 3, 3, dtype=dtype, device=dev), torch.zeros(1, dtype=dtype, device=dev)
    for where in ((0, 0, 0), (n1 - 1, 0, n3 // 2), (n1 - 1, n2 - 1, n3 - 1), (0, n2 - 1, 0), (n1 // 2, n2 // 2, n3 - 1)):
        img = base.clone()
        img[(1,) + where] = value
        _, ybar = K.sm_linear(img.to(dev), w, b)
        got, ref = ybar.cpu().double().view(2, 27), _patch(base)
        # v = where - e lies in the grid for the offsets that include the cell
        reads = torch.tensor([all(0 <= a - e < n for a, e, n in zip(where, d, shape)) for d in OFFSETS])
        assert torch.allclose(got[0], ref[0], rtol=2.0 ** -23, atol=0)
        assert torch.allclose(got[1][~reads], ref[1][~reads], rtol=2.0 ** -23, atol=2.0 ** -45)
        if value > 1e30:
            assert torch.allclose(got[1][reads], torch.full((1,), value / img[0].numel(), dtype=torch.float64), rtol=1e-6)
        else:
            assert not torch.isfinite(got[1][reads]).any()
