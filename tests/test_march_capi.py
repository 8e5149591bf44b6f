"""What the marching loops' C entries refuse, on the host, before any device call."""
import ctypes

import pytest

from seistorch_amd import _lib


@pytest.mark.parametrize("n", [-1, 0, (1 << 20) + 1, 1 << 62])
def test_batch_workspace_refuses_a_bad_count(n):
    shape = (ctypes.c_int64 * 6)(200, 300, 4, 500, 300, 1)
    assert _lib.load().seis_acoustic_march_batch_workspace(n, shape, 0, 0) == -1
    assert _lib.load().seis_acoustic_march_batch_workspace(1, None, 0, 0) == -1
    assert _lib.load().seis_acoustic_march_batch_workspace(1, shape, 0, 0) > 0


def test_forward_refuses_a_ring_whose_columns_share_a_lane():
    p = ctypes.c_void_p(4096)
    four = (ctypes.c_void_p * 4)(4096, 8192, 12288, 16384)
    last = (ctypes.c_int32 * 2)()
    for nx in (101, 102):
        with pytest.raises(RuntimeError, match="too small"):
            _lib.call("seis_acoustic_march_forward", p, p, p, 10, p, None, 0, None, 0, None, p,
                      None, 0, p, four, last, 1, 120, nx, 1e-3, 10.0, 49, 0, 0, 0, 0, None)
        shape = (ctypes.c_int64 * 6)(120, nx, 1, 10, 0, 0)
        dt_h = (ctypes.c_float * 2)(1e-3, 10.0)
        with pytest.raises(RuntimeError, match="too small"):
            _lib.call("seis_acoustic_march_batch_forward", 1, shape, dt_h, p, p, p, p, p, None,
                      None, p, None, 0, p, four, 49, 0, 0, None)
