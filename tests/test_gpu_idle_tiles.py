"""BF16 plans inside the solver leave out tiles without fluid: the solve must be the one that an
application of the plan on the whole grid gives."""
import numpy as np
import pytest
import torch

from mlpcg_amd import scenes as S

pytestmark = pytest.mark.gpu


def _flags(shape, case, seed):
    rng = np.random.default_rng(seed)
    f = np.full(shape, 3, dtype=np.int8)
    n1, n2, n3 = shape
    if case == "layer":      # whole idle tiles above, fluid up to a tile's last cell
        f[:, :, :64] = 2
    elif case == "halo":     # one more layer: the tile above has fluid in its halo only
        f[:, :, :65] = 2
        f[: n1 // 2, :, 64] = 3
    elif case == "corner":   # single cells beside the corners of tiles
        f[1:7, 1:7, 1:63] = 2
        for _ in range(12):
            i, j, k = (int(rng.integers(0, n // s)) * s for n, s in zip(shape, (2, 8, 64)))
            f[max(i - 1, 1), max(j - 1, 1), max(k - 1, 1)] = 2
    f[rng.random(shape) < 0.03] = 1
    for d in range(3):
        idx = [slice(None)] * 3
        for e in (0, -1):
            idx[d] = e
            f[tuple(idx)] = 0
    return f


@pytest.mark.parametrize("method", ["npsd", "npcg", "npcg_flex"])
@pytest.mark.parametrize("case", ["layer", "halo", "corner"])
@pytest.mark.parametrize("shape", [(48, 64, 128), (72, 32, 192)])
def test_solver_steps_match_plan_applications(dev, shape, case, method):
    from mlpcg_amd.sm_model_3d import SmallSMModelDn3D
    from mlpcg_amd.solver import FusedPCG
    print(f"idle tiles {shape} {case} {method}", flush=True)
    flags = _flags(shape, case, 4)
    fluid = np.flatnonzero(flags.ravel() == 2)
    open_ = np.pad((flags >= 2).astype(np.float32), 1)
    nb = sum(np.roll(open_, s, a) for a in range(3) for s in (-1, 1))[1:-1, 1:-1, 1:-1]
    img = torch.as_tensor((nb / 6 * (flags == 2)).astype(np.float32)[None], device=dev)
    torch.manual_seed(3)
    plan = SmallSMModelDn3D(3, 1, "trilinear").cuda().make_preconditioner(img, torch.bfloat16, fused_mode=2)
    assert plan.fused_blocks > 0 and fluid.size
    s = FusedPCG(flags, device=dev)
    b = torch.zeros(flags.size, device=dev)
    b[torch.as_tensor(fluid, device=dev)] = torch.randn(fluid.size, generator=torch.Generator().manual_seed(1)).to(dev)
    # the first step of every method moves along z = P(b / |b|), masked, x = alpha z with one
    # rounding.  npsd's first step runs the kernels of a masked application, so only roundings
    # of the ratios are left; the others' last block also sums dot products and takes the bias
    # as two FP16 parts (2^-22), which flips the BF16 rounding of about one tap in 2^13 by 2^-8:
    # sqrt(2^-13) 2^-8 = 2^-14.5 in the norm, more where taps cancel
    mask = torch.as_tensor((flags == 2).ravel(), device=dev)
    scale = 1.0 / b.double().norm().reshape(1)
    z = plan.apply(b, in_scale=scale, out_mask=mask.to(torch.uint8))
    k = int(z.abs().argmax())
    for again in (0, 1):  # whatever other applications left in the plan's buffers in between
        x, _ = s.solve(b, plan, method=method, max_it=1, tol=1e-12)
        assert torch.all(x[~mask] == 0)
        d = x / x[k] - z / z[k]
        if method == "npsd":
            assert float(d.abs().max()) <= 5 * 2.0 ** -24
        else:
            assert float(d.double().norm() / (z / z[k]).double().norm()) <= 2.0 ** -10
        plan.apply(torch.randn(flags.size, device=dev))
