"""The matrix-free solver on grids that are mostly air: runs of cells without fluid are skipped,
so nothing may be left in them from a caller's x0 or an earlier solve."""
import numpy as np
import pytest
import torch

from mlpcg_amd import scenes as S
from oracle import solvers as O

pytestmark = pytest.mark.gpu


def _flags(shape, seed):
    """Fluid in a few blobs and single cells, one of them beside every edge of a run."""
    rng = np.random.default_rng(seed)
    f = np.full(shape, 3, dtype=np.int8)
    for d in range(3):
        idx = [slice(None)] * 3
        for e in (0, -1):
            idx[d] = e
            f[tuple(idx)] = 0
    inner = f[1:-1, 1:-1, 1:-1]
    inner[rng.random(inner.shape) < 0.1] = 2
    inner[: inner.shape[0] // 2, :, : max(2, inner.shape[2] // 3)] = 2
    inner[rng.random(inner.shape) < 0.05] = 1
    return f


@pytest.mark.parametrize("method", ["npcg", "npcg_flex", "npsd"])
@pytest.mark.parametrize("shape", [(9, 10, 260), (7, 11, 34), (6, 9, 33), (12, 5, 16)])
@pytest.mark.parametrize("graphs", [False, True])
def test_air_is_skipped_and_stays_zero(dev, shape, method, graphs):
    from mlpcg_amd.solver import FusedPCG
    print(f"air {shape} {method} graphs={graphs}", flush=True)
    flags = _flags(shape, 1)
    fluid = np.flatnonzero(flags.ravel() == 2)
    air = torch.as_tensor(np.setdiff1d(np.arange(flags.size), fluid))
    A = S.build_matrix(flags)
    b = np.random.default_rng(2).standard_normal(fluid.size)
    b = A @ b
    s = FusedPCG(flags, device=dev, graphs=graphs)
    bv = s.vector(b)
    x1, i1 = s.solve(bv, method=method, max_it=400, tol=1e-5, history=True)
    ref = {"npcg": O.npcg, "npcg_flex": O.npcg_flex, "npsd": O.npsd}[method]
    h = ref(b, A, np.zeros_like(b), lambda r: r.copy(), 400, tol=1e-5)[2]
    # the first steps follow the FP64 loop to the FP32 rounding of the vectors
    m = min(4, len(h), len(i1["history"]))
    assert np.allclose(i1["history"][:m], h[:m], rtol=1e-4)
    xs = x1.cpu().numpy().ravel()[fluid].astype(np.float64)
    assert np.linalg.norm(b - A @ xs) <= 2e-5 * np.linalg.norm(b)
    assert torch.all(x1.cpu().ravel()[air] == 0)
    # a starting vector with values in the air: they act as boundary values of the first two
    # steps and are gone from every later iterate
    x0 = torch.as_tensor(np.random.default_rng(3).standard_normal(flags.size).astype(np.float32), device=dev)
    for it in (1, 2, 3):
        x, _ = s.solve(bv, x0=x0, method=method, max_it=it, tol=1e-12)
        assert torch.all(x.cpu().ravel()[air] == 0)
    # and nothing of it is left for the next solve
    x2, i2 = s.solve(bv, method=method, max_it=400, tol=1e-5)
    assert torch.equal(x1, x2) and i1["iters"] == i2["iters"]
