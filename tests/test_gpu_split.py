"""FP32 blocks on the matrix cores (split FP16 operands) against the FP64 oracle at the edges
of their tiles (64 z cells, 8 rows, 2 or 4 planes), for every channel count, odd and even
batches, images and weights far from 1, and the epilogues of a plan."""
import pytest
import torch

from oracle import model as M

pytestmark = pytest.mark.gpu

SHAPES = [(32, 32, 32), (7, 9, 300), (33, 17, 65), (5, 64, 64), (16, 15, 129), (64, 8, 63)]  # >= 2^14 voxels


def _inputs(C, B, shape, kind, seed):
    g = torch.Generator().manual_seed(seed)
    img = torch.rand(C, *shape, generator=g)
    x = torch.randn(B, 1, *shape, generator=g)
    bound = (27 * C) ** -0.5
    w = (torch.rand(27, C, 3, 3, 3, generator=g) * 2 - 1) * bound
    b = (torch.rand(27, generator=g) * 2 - 1) * bound
    if kind == "flags":  # exact in one FP16 value
        img = (img > 0.4).float()
    elif kind == "large":
        img = img * 3e7
    elif kind == "small":  # far below FP16, no bias to hide behind
        img, w, b = img * 1e-11, w * 1e-9, b * 0
    elif kind == "mixed":  # one voxel dwarfs the others; x vanishes in half of the grid
        img[0, shape[0] // 2, 3, 5] = 4e4
        x[..., shape[2] // 2:] = 0
    return img, x, w, b


def _bound(img, x, w, b):
    """|error| of y in units of A = sum_p (sum |W||img| + |b_p|) |x_p|.  Two FP16 values hold
    a number to 2^-23, and W_lo img_lo is left out: 2^-21 per product.  FP32 sums: at most 64
    roundings in K (6 matrix products per channel half, their inner sums), 32 in y.  Below
    FP16's denormals 2^-24 of values scaled to 2^4: 2^-28 of the largest W times image."""
    a = M.sm_block(img.abs(), x.abs(), w.abs(), b.abs())
    floor = 27 * 27 * img.shape[0] * 2.0 ** -27 * float(w.abs().max() * img.abs().max() * x.abs().max())
    return a * (2.0 ** -21 + 96 * 2.0 ** -24) + floor


@pytest.mark.parametrize("kind", ["random", "flags", "large", "small", "mixed"])
@pytest.mark.parametrize("C,B", [(1, 1), (2, 3), (3, 2)])
@pytest.mark.parametrize("shape", SHAPES)
def test_split_forward_vs_oracle(dev, shape, C, B, kind):
    from mlpcg_amd import kernels as K
    print(f"split forward {shape} C={C} B={B} {kind}", flush=True)
    img, x, w, b = _inputs(C, B, shape, kind, 5)
    y = K.sm_block_forward(img.to(dev), x.to(dev), w.to(dev), b.to(dev)).cpu().double()
    img, x, w, b = (t.double() for t in (img, x, w, b))
    err = (y - M.sm_block(img, x, w, b)).abs()
    assert torch.all(err <= _bound(img, x, w, b)), float((err / _bound(img, x, w, b)).max())


def test_split_forward_keeps_non_finite_values_local(dev):
    """An infinite or NaN x or image cell reaches the 27 (125) voxels whose stencils read it
    and no other; a zero x tile does not hide it."""
    from mlpcg_amd import kernels as K
    shape = (12, 24, 130)
    img, x, w, b = _inputs(1, 1, shape, "random", 6)
    for target, reach, zero_x in (("x", 1, False), ("img", 2, False), ("img", 2, True)):
        for bad in (float("inf"), float("nan")):
            im, xx = img.clone(), x.clone()
            if zero_x:
                xx.zero_()
            (xx[0, 0] if target == "x" else im[0])[5, 11, 64] = bad
            y = K.sm_block_forward(im.to(dev), xx.to(dev), w.to(dev), b.to(dev)).cpu()[0, 0]
            want = torch.zeros(shape, dtype=torch.bool)
            want[5 - reach:6 + reach, 11 - reach:12 + reach, 64 - reach:65 + reach] = True
            got = ~torch.isfinite(y)
            assert not torch.any(got & ~want), (target, bad)
            if target == "x" or not zero_x:
                assert bool(got[5, 11, 64]), (target, bad)
            else:
                assert bool(got.any())


@pytest.mark.parametrize("C,mask,swap,n,shape", [(1, False, False, 2, (64, 64, 68)), (3, True, False, 1, (66, 62, 72)),
                                                 (2, False, True, 1, (64, 72, 64)), (3, False, False, 2, (36, 100, 84))])
def test_split_plan_matches_stored_stencils(dev, C, mask, swap, n, shape):
    """Plans whose level 0 is above 2^18 voxels (fused_mode 2 recomputes K there for any channel
    count): with the output mask, the input scale and the
    pooled epilogue against the stored-stencil plan of the same model (fused_mode 0)."""
    from mlpcg_amd.sm_model_3d import SmallSMModelDn3D
    print(f"split plan {shape} C={C}", flush=True)
    torch.manual_seed(3)
    m = SmallSMModelDn3D(n, C, "trilinear", mask, swap).to(dev)
    g = torch.Generator().manual_seed(4)
    img = (torch.rand(C, *shape, generator=g) > 0.3).float().to(dev)
    r = torch.randn(*shape, generator=g).to(dev)
    scale = torch.tensor(0.37, dtype=torch.float64, device=dev)
    out = (torch.rand(*shape, generator=g) > 0.4).to(torch.uint8)
    out[:, :, 60:] = 0
    out = out.to(dev)
    a, b = m.make_preconditioner(img, fused_mode=2), m.make_preconditioner(img, fused_mode=0)
    assert a.nbytes < b.nbytes
    for args in ((None, None), (scale, out)):
        za, zb = a.apply(r, *args), b.apply(r, *args)
        # both FP32, roundings in another order: a few hundred half-ulps of the largest value
        assert float((za - zb).abs().max()) <= 300 * 2.0 ** -24 * float(zb.abs().max())
    x = torch.randn(*shape, generator=g).to(dev)
    ya, yb = a.apply_block(0, x, in_scale=scale), b.apply_block(0, x, in_scale=scale)
    assert float((ya - yb).abs().max()) <= 300 * 2.0 ** -24 * float(yb.abs().max())


@pytest.mark.parametrize("method", ["npcg", "npcg_flex", "npsd"])
def test_split_solve_matches_stored_stencils(dev, method):
    """The solver with its dot products in the last block's epilogue (FP32, 128 x 64 x 64)."""
    import numpy as np
    from mlpcg_amd import scenes as S
    from mlpcg_amd.sm_model_3d import SmallSMModelDn3D
    from mlpcg_amd.solver import FusedPCG
    torch.manual_seed(2)
    flags = np.full((128, 64, 64), S.FLUID, dtype=np.int8)
    flags[:, :, 40:] = S.AIR
    flags[40:60, 20:40] = S.SOLID
    for d in range(3):
        for e in (0, -1):
            np.moveaxis(flags, d, 0)[e] = S.BOUNDARY
    m = SmallSMModelDn3D(3, 1).to(dev)
    img = torch.as_tensor(S.image_channels(flags, 1), device=dev)
    solver = FusedPCG(flags, device=dev)
    b = solver.vector(S.make_rhs(flags, 1)[0])
    xs = []
    for mode in (1, 0):
        plan = m.make_preconditioner(img, fused_mode=mode)
        xs.append(solver.solve(b, plan, method=method, max_it=6, tol=1e-30, history=True))
    (xa, ia), (xb, ib) = xs
    # six iterations of the same recurrence: FP32 preconditioners equal to a few 1e-7
    assert np.allclose(ia["history"], ib["history"], rtol=1e-4)
    assert float((xa - xb).norm() / xb.norm()) < 1e-4
