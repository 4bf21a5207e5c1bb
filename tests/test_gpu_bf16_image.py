"""BF16 block forwards convert their image as they stage it: the same values as from an FP16 copy
of the image handed in."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [1, 2, 3])
@pytest.mark.parametrize("shape", [(64, 64, 64), (72, 32, 128), (128, 128, 192)])
def test_image_converted_in_the_kernel(dev, C, shape):
    from mlpcg_amd import kernels as K
    from mlpcg_amd._lib import check, lib, ptr, stream_ptr
    print(f"bf16 image {shape} C={C}", flush=True)
    gen = torch.Generator().manual_seed(6)
    img = torch.rand(C, *shape, generator=gen).to(torch.bfloat16).to(dev)
    x = torch.randn(1, 1, *shape, generator=gen).to(torch.bfloat16).to(dev)
    w, b = torch.randn(27, C, 3, 3, 3, generator=gen).to(dev), torch.randn(27, generator=gen).to(dev)
    y = K.sm_block_forward(img, x, w, b)
    copy, z = img.to(torch.float16), torch.empty_like(x)
    n = lib.mlpcg_sm_block_workspace_size(C, 1, *shape, 3)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)
    check(lib.mlpcg_sm_block_forward_ex(ptr(img), ptr(copy), None, ptr(x), ptr(w), ptr(b), ptr(z), ptr(ws), C, 1, *shape, 3,
                                        stream_ptr(x.device)))
    assert torch.equal(y, z)
