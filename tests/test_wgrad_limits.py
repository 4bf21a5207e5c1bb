"""The weight gradient's launcher refuses tensors that its 32-bit offsets do not reach (the entry
points' own limit on the grid lies below)."""
import ctypes


def test_weight_gradient_refuses_tensors_of_two_gigabytes():
    from mlpcg_amd import _lib
    fn = _lib.lib._ZN5mlpcg12launch_wgradEiPKvS1_S1_PfiiiiiiP12ihipStream_t
    fn.restype = ctypes.c_int
    for dtype, grid in ((1, (4, 16384, 8192)), (3, (2, 32768, 16384)), (2, (1, 1 << 15, 1 << 15))):
        assert fn(dtype, None, None, None, None, 1, 1, 1, *grid, None) == -1
        assert b"too large" in _lib.lib.mlpcg_last_error()
    # the entry points: 27 V below 2^33
    for dtype in range(4):
        args = [None, None, None, None, None, None, None, None, None, 1, 1, 1 << 10, 1 << 10, 304, dtype, None]
        assert _lib.lib.mlpcg_sm_block_backward(*args) == -1
        assert b"too large" in _lib.lib.mlpcg_last_error()
