"""Two SM linears of one image in one call (a level's c0 and c1) against two single calls."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.bfloat16])
@pytest.mark.parametrize("C,shape", [(1, (1, 1, 1)), (3, (5, 6, 7)), (2, (16, 16, 16)), (3, (40, 33, 66))])
def test_pair_equals_single_calls(dev, dtype, C, shape):
    from mlpcg_amd import kernels as K
    img = torch.rand(C, *shape, device=dev).to(dtype)
    ws = [(torch.randn(1, C, 3, 3, 3, device=dev), torch.randn(1, device=dev)) for _ in range(2)]
    z = K.sm_linear_pair(img, *ws[0], *ws[1])
    for (w, b), zi in zip(ws, z):
        assert torch.equal(zi, K.sm_linear(img, w, b)[0]) and zi.shape == (1,)


@pytest.mark.parametrize("swap", [False, True])
def test_eval_forward_keeps_overrides(dev, swap):
    """eval_forward takes the pair for plain modules and calls what a user put in their place."""
    from mlpcg_amd.sm_model_3d import SmallSMModelDn3D
    torch.manual_seed(1)
    m = SmallSMModelDn3D(2, 1, "trilinear", False, swap).to(dev)
    img, b = torch.rand(1, 16, 16, 24, device=dev), torch.randn(1, 1, 16, 16, 24, device=dev)
    with torch.no_grad():
        c0, c1 = [], []
        y = m.eval_forward(img, b, None, [], c0, c1)
        ref = m.eval_forward(img, b, None, [], [c.clone() for c in c0], [c.clone() for c in c1])
        assert torch.equal(y, ref) and len(c0) == len(c1) == 2
        calls = []
        old = m.c1[0].eval_forward
        m.c1[0].eval_forward = lambda image, timer=None: (calls.append(1), old(image, timer) * 2)[1]
        d0, d1 = [], []
        m.eval_forward(img, b, None, [], d0, d1)
        assert calls == [1] and torch.equal(d1[0], c1[0] * 2) and torch.equal(d0[0], c0[0]) and torch.equal(d1[1], c1[1])


def test_stream_handle_follows_the_current_stream(dev):
    from mlpcg_amd._lib import stream_ptr
    s = torch.cuda.Stream()
    d = torch.zeros(1, device=dev).device
    assert stream_ptr(d) == torch.cuda.current_stream(d).cuda_stream
    with torch.cuda.stream(s):
        assert stream_ptr(d) == s.cuda_stream == stream_ptr() == stream_ptr(torch.device("cuda"))
