"""Mean patch of a grid of more than 2^32 z-runs (a plan's image may be that large; the block
entry points refuse it): cells beyond the 2^32nd are counted, and the neighbours of the count's
end."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def test_more_than_2_32_runs(dev):
    from mlpcg_amd import _lib
    n1 = n2 = 65537  # 2^32 + 131073 cells, one to a run
    if torch.cuda.mem_get_info()[0] < 16 << 30:
        pytest.skip("needs 16 GB of device memory")
    img = torch.zeros(n1, n2, 1, dtype=torch.bfloat16, device=dev)
    marks = {(0, 0): 1.0, (65535, 65536): 2.0, (65536, 5): 4.0, (65536, 65536): 8.0, (40000, 1): 16.0}
    for at, v in marks.items():
        img[at] = v
    w, b = torch.zeros(27, device=dev), torch.zeros(1, device=dev)
    z, ybar = torch.empty(1, device=dev), torch.empty(27, device=dev)
    work = torch.empty(512 * 27 * 8, dtype=torch.uint8, device=dev)
    fn = _lib.lib._ZN5mlpcg16launch_sm_linearEiPKvS1_S1_PvS2_S2_iiiiP12ihipStream_t
    fn.restype = ctypes.c_int
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    print("mean patch 65537 x 65537 x 1", flush=True)
    assert fn(3, p(img), p(w), p(b), p(z), p(ybar), p(work), 1, n1, n2, 1, ctypes.c_void_p(_lib.stream_ptr(dev))) == 0
    got = ybar.cpu().double() * (n1 * n2)
    for k in range(27):
        d = (k // 9 - 1, k // 3 % 3 - 1)
        want = sum(v for (i, j), v in marks.items() if 0 <= i - d[0] < n1 and 0 <= j - d[1] < n2) if k % 3 == 1 else 0.0
        assert abs(float(got[k]) - want) <= 1e-6 * max(want, 1.0), (k, float(got[k]), want)
