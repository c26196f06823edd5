"""Reductions over every axis at the edges of the kernels' rules (short rows
sharing a wave, long rows of odd length or other types, strips, chunks and one
lane per output along the columns), through the C ABI, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (outer, len, inner).  Rows: units per row around 8, 16, 32 and the wave
# kernels; long rows of every alignment, few enough to split.
ROWS = [(n, length, 1) for n, length in
        [(1, 1), (5, 7), (65, 8), (1000, 9), (33, 31), (70, 33), (9, 100), (129, 128), (7, 132),
         (3, 2047), (3, 2048), (2, 2049), (1, 4099), (5, 8192), (2100, 2050), (1, 200003)]]
# Columns: strips of one to many units, row groups that do not divide 256,
# short and long axes (chunked above 4096), slices of at most 128 units.
COLS = [(1, 3, 2), (300, 8, 2), (4, 8, 16), (4, 9, 16), (70, 197, 12), (5, 197, 768), (3, 64, 260),
        (1, 4096, 4), (1, 4097, 4), (1, 16385, 3), (2, 5000, 5), (1, 70, 1027), (1, 1, 9),
        (300, 5, 4096), (1, 20000, 130)]
DT = {"f32": np.float32, "f64": np.float64, "i32": np.int32, "i64": np.int64, "i16": np.int16, "bool": np.bool_}


def _data(dt, shape, seed):
    rng = np.random.default_rng(seed)
    if dt == "bool":
        return rng.random(shape) < 0.3
    if dt.startswith("i"):
        return rng.integers(-1000, 1000, shape).astype(DT[dt])
    return rng.standard_normal(shape).astype(DT[dt])


@pytest.mark.parametrize("shape", ROWS + COLS, ids=str)
@pytest.mark.parametrize("dt", sorted(DT))
def test_reduce_shapes(hip, dt, shape):
    a = _data(dt, shape, sum(shape))
    d = hip.DeviceBuffer.from_numpy(a)
    for op in ("max", "min"):
        got = hip.reduce(op, d, 1).numpy()
        assert np.array_equal(got, getattr(a, op)(axis=1, keepdims=True)), op
    got = hip.reduce("sum", d, 1).numpy()
    if dt == "bool":
        assert np.array_equal(got, a.any(axis=1, keepdims=True))
    elif dt.startswith("i"):
        assert np.array_equal(got, a.sum(axis=1, keepdims=True, dtype=np.int64).astype(a.dtype))
    else:
        # A term passes through at most ceil(len / 32) additions of its
        # accumulator (a lane's loop, 8 accumulators x 4 row groups or more,
        # fewer where the axis is split), then a few more to join them.
        u = np.finfo(a.dtype).eps / 2
        mag = np.abs(a).astype(np.float64).sum(axis=1, keepdims=True)
        want = a.astype(np.longdouble).sum(axis=1, keepdims=True)
        depth = shape[1] // 32 + 40
        assert np.all(np.abs(got - want) <= depth * u * mag)


@pytest.mark.parametrize("shape", [(70, 24, 1), (3, 2051, 1), (5, 197, 12), (1, 5000, 6)], ids=str)
def test_reduce_extremes(hip, shape):
    """Values at the ends of the type, infinities and NaN where every kernel
    has an identity or an idle lane: max and min skip NaN as std::max from the
    identity does, an all -inf row gives the lowest finite value."""
    a = _data("f32", shape, 3)
    a[0, :, 0] = -np.inf
    a[0, shape[1] // 2, 0] = np.nan
    a[-1, -1, -1] = np.inf
    d = hip.DeviceBuffer.from_numpy(a)
    low = np.finfo(np.float32).min
    want = np.fmax.reduce(a, axis=1, initial=low, keepdims=True)
    assert np.array_equal(hip.reduce("max", d, 1).numpy(), want)
    want = np.fmin.reduce(a, axis=1, initial=-low, keepdims=True)
    assert np.array_equal(hip.reduce("min", d, 1).numpy(), want)


@pytest.mark.parametrize("shape", [(256, 3001), (1000, 2049), (64, 32767), (3, 32768 * 2 + 1), (4, 200001), (1, 1000003)],
                         ids=str)
@pytest.mark.parametrize("dt", ["f32", "f64", "i32"])
def test_long_rows_in_parts(hip, dt, shape):
    """Long rows that are not fp32 float4s: one launch until a second part has 64
    units a lane, then parts whose results are a row of their own.  The sums of
    positive values: a lane's chain is 2^-10 of the row or less, so what rounds is
    the joins, each level half the one after it (0.58 half-ulps rms times sqrt 2,
    and a second set for the parts)."""
    import ctypes as C
    a = _data(dt, shape, sum(shape))
    a = np.abs(a)
    d = hip.DeviceBuffer.from_numpy(a.reshape(shape + (1,)))
    n0, n1 = C.c_uint64(), C.c_uint64()
    hip.check(hip.lib().lmp_rt_kernel_launch_count(C.byref(n0)))
    got = hip.reduce("sum", d, 1).numpy().reshape(-1)
    hip.check(hip.lib().lmp_rt_kernel_launch_count(C.byref(n1)))
    assert n1.value - n0.value == (1 if shape[1] < 2 * 64 * 256 else 2)
    if dt == "i32":
        assert np.array_equal(got, a.sum(axis=1, dtype=np.int64).astype(np.int32))
        return
    want = a.astype(np.longdouble).sum(axis=1)
    u = np.finfo(a.dtype).eps / 2
    err = np.abs((got - want) / want).astype(np.float64)
    # up to four outputs: the root mean square of as few is under twice the expected
    bound = 0.58 * np.sqrt(2 * (1 if n1.value - n0.value == 1 else 2)) * u
    assert np.sqrt(np.mean(err ** 2)) <= bound * (1.15 if shape[0] >= 64 else 2)


# The columns' rules at their edges: a lane per output for short axes and few
# units, a workgroup a slice from three and a half values a lane on, strips that
# end inside a 128-byte line or leave a short last one, power of two widths,
# strips of single values of 1 KiB and less, one pass up to 256 KiB a workgroup
# and down to a line (whole lines) or two (others), 512-byte and 256-byte strips
# in parts, 65535 outer slices and more.
MORE_COLS = [(300, 1, 300), (2100, 16, 64), (2100, 17, 64), (8200, 40, 3), (2800, 32, 8), (3, 33, 8), (2, 200, 130),
             (1, 300, 1544), (5, 300, 600), (29, 2752, 24), (1, 3000, 256), (2, 130, 1100), (6, 700, 1027),
             (1, 896, 8192), (1, 192, 6400), (3, 500, 2500), (4, 4200, 512), (1, 4200, 2304), (49, 777, 48),
             (2600, 18, 51), (2600, 17, 51), (2100, 64, 63),
             (65535, 5, 6), (65536, 5, 6), (65535, 33, 20)]


@pytest.mark.parametrize("shape", MORE_COLS, ids=str)
@pytest.mark.parametrize("dt", ["f32", "f64", "i32", "i16", "bool"])
def test_reduce_column_rules(hip, dt, shape):
    test_reduce_shapes(hip, dt, shape)


@pytest.mark.parametrize("shape,launches", [((1, 3000, 256), 1), ((6, 3937, 64), 1), ((1, 3111, 1024), 1),
                                            ((1, 896, 8192), 1), ((1, 4096, 4096), 2)], ids=str)
def test_column_sums_in_one_pass(hip, shape, launches):
    """A short axis of small slices in one launch; the sums' joins (0.58 half-ulps
    rms a level, six or fewer count) bound the error of positive values."""
    import ctypes as C
    a = np.abs(_data("f32", shape, 5)) + np.float32(0.5)
    d = hip.DeviceBuffer.from_numpy(a)
    n0, n1 = C.c_uint64(), C.c_uint64()
    hip.check(hip.lib().lmp_rt_kernel_launch_count(C.byref(n0)))
    got = hip.reduce("sum", d, 1).numpy()
    hip.check(hip.lib().lmp_rt_kernel_launch_count(C.byref(n1)))
    assert n1.value - n0.value == launches
    want = a.sum(axis=1, keepdims=True, dtype=np.float64)
    assert np.linalg.norm(got - want) <= 0.58 * np.sqrt(6) * 2.0 ** -24 * np.linalg.norm(want)
