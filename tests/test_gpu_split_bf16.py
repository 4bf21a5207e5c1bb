"""BF16 block forwards on grids and batches that the fused apply does not take, against FP64 at
the edges of the tiles (64 z cells, 8 rows, 2 or 4 planes)."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,B,shape", [(1, 1, (4, 64, 65)), (2, 3, (33, 21, 31)), (3, 2, (17, 40, 63)), (1, 2, (128, 64, 64)),
                                       (1, 5, (130, 128, 1)), (3, 1, (9, 31, 193)), (1, 2, (134, 130, 129)), (3, 2, (128, 65, 130))])
def test_bf16_block_forward(dev, C, B, shape):
    from mlpcg_amd import kernels as K
    print(f"bf16 forward C={C} B={B} {shape}", flush=True)
    gen = torch.Generator().manual_seed(7)
    img = torch.rand(C, *shape, generator=gen).to(torch.bfloat16).to(dev)
    x = torch.randn(B, 1, *shape, generator=gen).to(torch.bfloat16).to(dev)
    w = ((torch.rand(27, C, 3, 3, 3, generator=gen) - 0.5) * 0.4).to(dev)
    b = ((torch.rand(27, generator=gen) - 0.5) * 0.4).to(dev)
    y = K.sm_block_forward(img, x, w, b)[:, 0].double()

    def shifts(t):
        p = torch.nn.functional.pad(t, (1, 1, 1, 1, 1, 1))
        return [p[..., 1 + d[0]:1 + d[0] + shape[0], 1 + d[1]:1 + d[1] + shape[1], 1 + d[2]:1 + d[2] + shape[2]]
                for d in itertools.product((-1, 0, 1), repeat=3)]

    P = torch.cat([s[:, None] for s in shifts(img.double())], 1).flatten(0, 1).flatten(1)
    W = w.double().reshape(27, -1)
    ref, mag = torch.zeros_like(y), torch.zeros_like(y)
    for p, xs in enumerate(shifts(x.double()[:, 0])):
        ref += ((W[p] @ P).reshape(shape) + b.double()[p]) * xs
        mag += ((W[p].abs() @ P).reshape(shape) + b.double()[p].abs()) * xs.abs()
    # room for weights of 11 bits (2^-12), FP32 sums, the result rounded to BF16 (2^-9)
    assert torch.all((y - ref).abs() <= mag * (2.0 ** -12 + 64 * 2.0 ** -24) + ref.abs() * 2.0 ** -8)
    assert float((y - ref).norm() / ref.norm()) <= 2.0 ** -8
