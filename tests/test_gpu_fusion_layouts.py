"""Fused kernels over every layout of their plans against the eager kernels,
bit for bit: outputs whose rows are not whole 16-byte units, broadcasts over
any axes, float64, and row regions of long rows (a workgroup per row, split as
the eager reductions split them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rsl(hip):
    import rushlite_amd
    return rushlite_amd


def _vars(rsl, shapes, dt, seed, grad=False):
    rng = np.random.default_rng(seed)
    return [rsl.Variable((rng.standard_normal(s) + 1.5).astype(dt), requires_grad=grad,
                         dtype=getattr(rsl.dtype, dt)) for s in shapes]


def _same(a, b):
    assert a.shape == b.shape and a.dtype == b.dtype
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


# Small outputs (one value per lane), then sizes around one unit, rows of one to a few values (several row ends
# in a unit), odd rows, whole-unit rows under 3-d and 4-d broadcasts.
LAYOUTS = [((1,), (1,)), ((3,), (1,)), ((5,), (5,)), ((7, 1), (1, 3)), ((9, 3), (9, 1)), ((33, 5), (5,)),
           ((1, 2), (9, 1)), ((255, 7), (255, 1)), ((64, 130), (130,)), ((4, 1, 3), (1, 5, 3)), ((2, 3, 8), (3, 1)),
           ((5, 6, 8), (5, 1, 8)), ((3, 4, 12), (1, 4, 1)), ((2, 3, 4, 5), (3, 1, 5)), ((6, 1, 2, 1), (1, 5, 1, 4)),
           ((1001, 37), (1001, 37)), ((70, 4, 6), (70, 1, 6)), ((8003, 3), (8003, 1)), ((30001, 1), (1, 2)),
           ((4001, 7), (7,)), ((40, 1, 30), (1, 17, 30)), ((60, 17, 20), (60, 1, 20)), ((50, 3, 128), (3, 1)),
           ((3, 90, 2, 40), (90, 1, 40)), ((16385,), (1,)), ((20002,), (20002,))]


@pytest.mark.parametrize("sa,sb", LAYOUTS, ids=str)
@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_elementwise_layouts(rsl, sa, sb, dt):
    a, b = _vars(rsl, [sa, sb], dt, len(sa) * 7 + len(sb))

    def chain():
        t = a * b  # held by the caller: a second output of the kernel
        return t, rsl.exp(-t) * b - rsl.clamp(a, 0.5, 1e30) / (b + 1)

    with rsl.no_grad():
        want = [v.numpy() for v in chain()]
        with rsl.capture_on():
            t, y = chain()
        y.realize()
        _same(y.numpy(), want[1])
        _same(t.numpy(), want[0])


@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_grouped_updates_of_odd_sizes(rsl, dt):
    """realize_all over parameters of odd sizes runs their updates as one
    kernel of 16-byte units, the bits of the separate ones."""
    ps = _vars(rsl, [(10,), (3, 7), (1,), (64, 33)], dt, 5)
    gs = _vars(rsl, [(10,), (3, 7), (1,), (64, 33)], dt, 6)
    want = [(p.data - 0.01 * g.data).numpy() for p, g in zip(ps, gs)]
    with rsl.capture_on():
        new = [rsl.Variable(p.data - 0.01 * g.data) for p, g in zip(ps, gs)]
    s0 = rsl._stats()["fused_launches"]
    rsl.realize_all(new)
    assert rsl._stats()["fused_launches"] == s0 + 1
    for n, w in zip(new, want):
        _same(n.numpy(), w)


# Rows at the ends of the workgroup kernels: a wave's longest, one unit more or
# less than whole lanes, odd (single values), split over two and three parts
# by the eager reductions (few rows of 8192 and more), the longest, one past it.
ROWS = [((3, 2047), "float32"), ((3, 2048), "float32"), ((5, 2049), "float32"), ((4, 4100), "float32"),
        ((2100, 2052), "float32"), ((3, 8192), "float32"), ((700, 12292), "float32"), ((2, 16384), "float32"),
        ((2, 16383), "float32"), ((2, 16388), "float32"), ((2, 3, 2050), "float32"), ((3, 2048), "float64"),
        ((3, 2051), "float64"), ((2, 8190), "float64"), ((2, 8194), "float64")]


@pytest.mark.parametrize("shape,dt", ROWS, ids=str)
def test_long_rows_softmax_and_loss(rsl, shape, dt):
    """Softmax, the cross-entropy rows and their gradients, captured against
    eager."""
    axis = len(shape) - 1
    (x_np,) = [np.random.default_rng(shape[-1]).standard_normal(shape).astype(dt) * 3]
    y_np = np.zeros(shape, dt)
    y_np[..., 5] = 1

    def run(captured):
        x = rsl.Variable(x_np, requires_grad=True, dtype=getattr(rsl.dtype, dt))
        y = rsl.Variable(y_np, dtype=getattr(rsl.dtype, dt))
        with rsl.capture_on(captured):
            e = rsl.exp(x - rsl.max(x, axis))
            p = e / rsl.sum(e, axis)
            loss = rsl.sum(-y * rsl.log(p + 1e-3), axis)
        loss.backward()
        return p.numpy(), loss.numpy(), x.grad.numpy()

    want = run(False)
    for g, w in zip(run(True), want):
        _same(g, w)
    x64 = x_np.astype(np.float64)
    e64 = np.exp(x64 - x64.max(axis, keepdims=True))
    p64 = e64 / e64.sum(axis, keepdims=True)
    assert np.max(np.abs(want[0] - p64)) <= (1e-6 if dt == "float32" else 1e-14)


@pytest.mark.parametrize("op", ["sum", "max", "min", "prod"])
@pytest.mark.parametrize("shape,dt", [((3, 2056), "float32"), ((2, 9001), "float32"), ((2, 5000), "float64")], ids=str)
def test_long_rows_reductions_and_special_values(rsl, op, shape, dt):
    """Each reduction over a long fused row, with signed zeros, infinities and
    NaN in it, and elementwise work after it, captured against eager."""
    rng = np.random.default_rng(4)
    x_np = (1 + 0.001 * rng.standard_normal(shape)).astype(dt)
    x_np[1, ::7] = -0.0
    x_np[1, 3::11] = 0.0
    x_np[0, 5] = np.inf
    x_np[-1, 6] = np.nan if shape[0] > 2 else -np.inf
    (w,) = _vars(rsl, [(shape[1],)], dt, 9)
    x = rsl.Variable(x_np, dtype=getattr(rsl.dtype, dt))

    def f():
        return getattr(rsl, op)(x * 1.0, 1) / (x * x + 1.0) + w

    with rsl.no_grad():
        want = f().numpy()
        with rsl.capture_on():
            y = f()
        got = y.numpy()
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got[~nan].view(np.uint8), want[~nan].view(np.uint8))
