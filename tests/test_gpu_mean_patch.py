"""The SMLinear mean patch against the oracle where its reduction can go wrong: extents of 1
and 2 (a cell on two faces of one axis), odd extents, and both sides of the grid size at
which the one-workgroup kernel gives way to partial sums (4096 z-runs)."""
import pytest
import torch

from oracle import model as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("C,shape", [(1, (1, 1, 1)), (3, (1, 5, 2)), (2, (2, 1, 7)), (3, (3, 2, 4)), (1, (5, 7, 9)),
                                     (3, (16, 16, 64)), (3, (16, 17, 64)), (1, (33, 64, 62)), (2, (40, 64, 260))])
def test_mean_patch_sizes(dev, dtype, C, shape):
    from mlpcg_amd import kernels as K
    print(f"mean patch {dtype} C={C} {shape}", flush=True)
    g = torch.Generator().manual_seed(3)
    acc = torch.float64 if dtype == torch.float64 else torch.float32
    img = (torch.rand(C, *shape, generator=g, dtype=torch.float64) - 0.25).to(dtype)
    w = (torch.rand(1, C, 3, 3, 3, generator=g, dtype=torch.float64) - 0.5).to(acc)
    b = (torch.rand(1, generator=g, dtype=torch.float64) - 0.5).to(acc)
    z, ybar = K.sm_linear(img.to(dev), w.to(dev), b.to(dev))
    zr, yr = M.sm_linear(img.double(), w.double(), b.double())
    # FP64 sums: one rounding to the output type, and FP64 rounding of sums of |img| <= 1
    eps = 2.0 ** -52 if acc == torch.float64 else 2.0 ** -23
    tol = eps + 2.0 ** -45
    assert float((ybar.cpu().double() - yr).abs().max()) <= tol
    # z sums 27 C rounded entries with |w| <= 1/2, and is rounded once itself
    assert float((z.cpu().double() - zr).abs().max()) <= 14 * C * tol + eps * (1 + 14 * C)
