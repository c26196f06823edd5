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


def _ends(hip, buf, n, dtype):
    """A few values at the start, the middle and the end of n."""
    got = []
    for at in (0, n // 2, n - 8):
        x = np.zeros(8, dtype)
        hip.check(hip.lib().lmp_rt_memcpy_d2h(x.ctypes.data_as(C.c_void_p),
                                              C.c_void_p(buf.ptr + x.itemsize * at), x.nbytes))
        got.append(x)
    return np.concatenate(got)


@pytest.mark.parametrize("kind", ["int_gemm", "transpose", "thin_rows", "strided_column_sums"])
def test_matrix_kernels_past_a_grid(hip, kind):
    """One workgroup of 256 lanes per tile, row or block of columns, 2^32 threads
    or more in all: ones, so every result is the number of terms."""
    L, n = hip.lib(), {"thin_rows": (1 << 29) + 32, "strided_column_sums": (1 << 26) + 8}.get(kind, (1 << 30) + 64)
    t, code = {"int_gemm": (np.int16, hip.INT16), "transpose": (np.bool_, hip.BOOL)}.get(kind, (np.float32, hip.FLOAT32))
    rows = {"thin_rows": 4, "strided_column_sums": 8}.get(kind, 1)
    big, out = hip.DeviceBuffer((n, rows), t), hip.DeviceBuffer((n,), t)
    one = hip.DeviceBuffer.from_numpy(np.ones(8, t))
    hip.check(L.lmp_k_fill(code, big.ptr, n * rows, 1.0))
    hip.check(L.lmp_k_fill(code, out.ptr, n, 0.0))
    bufs = [big, out, one]
    if kind == "int_gemm":
        hip.check(L.lmp_k_gemm(code, 0, 0, n, 1, 1, big.ptr, 1, one.ptr, 1, out.ptr, 1, 0))
    elif kind == "transpose":
        hip.check(L.lmp_k_transpose(code, out.ptr, big.ptr, 1, n))
    elif kind == "thin_rows":
        hip.check(L.lmp_k_gemm_f32(0, 1, 1, n, 4, one.ptr, 4, big.ptr, 4, out.ptr, n, 0))
    else:
        sums = hip.DeviceBuffer((n,), t)
        bufs.append(sums)
        hip.check(L.lmp_k_fill(code, sums.ptr, n, 0.0))
        hip.check(L.lmp_k_gemm_colsum_f32(0, 1, 1, n, 4, one.ptr, 4, big.ptr, 8, out.ptr, n, 0, sums.ptr, 0))
        assert np.all(_ends(hip, sums, n, t) == 4)
    want = 4 if rows > 1 else 1
    assert np.all(_ends(hip, out, n, t) == want)
    for b in bufs:
        b.free()
    hip.check(L.lmp_rt_empty_cache())


@pytest.mark.parametrize("shape", [((1 << 32) + 8,), (1 << 16, 1 << 15)], ids=str)
def test_fused_chain_of_2_31_values_or_more(hip, shape):
    """A captured chain over 8 GiB or more runs on the float4 plan: marks around
    2^31, 2^32 and the ends come out at their own places, ones elsewhere."""
    import rushlite_amd as rsl
    n = int(np.prod([int(d) for d in shape], dtype=np.int64))
    with rsl.no_grad():
        a = rsl.ones(list(shape), device=rsl.device.hip, dtype=rsl.dtype.float32)
        base = rsl._storage_ptr(a.data)
        places = [p for p in (0, 4, (1 << 31) - 8, 1 << 31, (1 << 32) - 8, 1 << 32, n - 8) if 0 <= p <= n - 8]
        for i, p in enumerate(places):
            x = np.arange(8, dtype=np.float32) + 10 * (i + 1)
            hip.check(hip.lib().lmp_rt_memcpy_h2d(C.c_void_p(base + 4 * p), x.ctypes.data_as(C.c_void_p), 32))
        with rsl.capture_on():
            y = a * a + a
        assert "lmp_v4 o;" in rsl._fused_source(y)
        y.realize()
        want = np.ones(8, np.float32)
        for p in places + [n // 2 + 64, n - 64]:
            x, got = np.zeros(8, np.float32), np.zeros(8, np.float32)
            hip.check(hip.lib().lmp_rt_memcpy_d2h(x.ctypes.data_as(C.c_void_p), C.c_void_p(base + 4 * p), 32))
            hip.check(hip.lib().lmp_rt_memcpy_d2h(got.ctypes.data_as(C.c_void_p),
                                                  C.c_void_p(rsl._storage_ptr(y.data) + 4 * p), 32))
            assert np.array_equal(got, x * x + x), p
        assert np.array_equal(x, want)  # the last place is an unmarked one
    del a, y
    hip.check(hip.lib().lmp_rt_empty_cache())
