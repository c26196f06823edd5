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
