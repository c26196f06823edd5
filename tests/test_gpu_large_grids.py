"""One-shot launches whose work items would not fit a grid's 32-bit thread
count: fewer than 2^32 threads are launched and every element is written."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 32) + 5, (1 << 32) - 61], ids=str)
def test_scalar_kernels_past_a_grid(hip, n):
    """A bool fill and cast of n elements, one a lane: the ends and the middle."""
    L = hip.lib()
    a, out = hip.DeviceBuffer((n,), np.bool_), hip.DeviceBuffer((n,), np.int16)
    hip.check(L.lmp_k_fill(hip.BOOL, a.ptr, n, 1.0))
    hip.check(L.lmp_k_cast(hip.BOOL, hip.INT16, out.ptr, a.ptr, n))
    got = np.zeros(64, np.int16)
    for at in (0, n // 2, (1 << 31) - 32, n - 64):
        hip.check(L.lmp_rt_memcpy_d2h(got.ctypes.data_as(C.c_void_p), C.c_void_p(out.ptr + 2 * at), 128))
        assert np.all(got == 1), at
    a.free()
    out.free()
    hip.check(L.lmp_rt_empty_cache())


@pytest.mark.parametrize("rows,cols", [((1 << 26) + 3, 5), ((1 << 25) + 1, 33)], ids=str)
def test_row_sums_past_a_grid(hip, rows, cols):
    """Rows of ones (int16) beyond 2^32 threads of a wave per row."""
    L = hip.lib()
    a, out = hip.DeviceBuffer((rows, cols), np.int16), hip.DeviceBuffer((rows, 1), np.int16)
    hip.check(L.lmp_k_fill(hip.INT16, a.ptr, rows * cols, 1.0))
    hip.check(L.lmp_k_fill(hip.INT16, out.ptr, rows, 0.0))
    hip.check(L.lmp_k_reduce(hip.RED["sum"], hip.INT16, out.ptr, a.ptr, rows, cols, 1))
    assert np.all(out.numpy() == cols)
    a.free()
    out.free()
    hip.check(L.lmp_rt_empty_cache())
