"""fp32 products of up to 32 rows with B transposed: column blocks of 32 with
and without a split of K, edges of both, the epilogues and the no-allocation
entry."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# Fewer, as many and more blocks of 32 columns than CUs; K of one short tile,
# remainders of a workgroup's 128, splits whose last part is short or leaves
# waves without work; m of one, some and all rows.
SHAPES = [(32, 8, 8200), (1, 33, 4), (17, 100, 260), (31, 4098, 516), (32, 4224, 1000), (5, 1030, 4100),
          (32, 2048, 2052), (3, 8196, 132), (32, 8160, 388)]


@pytest.mark.parametrize("m,n,k", SHAPES, ids=str)
def test_thin_transposed_b(hip, m, n, k):
    rng = np.random.default_rng(m + n + k)
    L = hip.lib()
    up = hip.DeviceBuffer.from_numpy
    # small integers: every sum is exact in any order
    a = rng.integers(-8, 9, (m, k)).astype(np.float32)
    b = rng.integers(-8, 9, (n, k)).astype(np.float32)
    want = a @ b.T
    ap, bp = (np.full((x.shape[0], k + 4), np.nan, np.float32) for x in (a, b))
    ap[:, :k], bp[:, :k] = a, b
    da, db = up(ap), up(bp)
    bias = rng.integers(-8, 9, n).astype(np.float32)
    dbias = up(bias)
    for ldc in (n, n + 3):
        c0 = rng.integers(-8, 9, (m, ldc)).astype(np.float32)
        for entry in (L.lmp_k_gemm_f32, L.lmp_k_gemm_f32_noalloc):
            dc = up(c0)
            for acc in (1, 0):
                hip.check(entry(0, 1, m, n, k, da.ptr, k + 4, db.ptr, k + 4, dc.ptr, ldc, acc))
                got = dc.numpy()
                assert np.array_equal(got[:, :n], c0[:, :n] + want if acc else want)
                assert np.array_equal(got[:, n:], c0[:, n:])
        dc = up(c0)
        hip.check(L.lmp_k_linear_relu_f32(0, 1, m, n, k, da.ptr, k + 4, db.ptr, k + 4, dbias.ptr, dc.ptr, ldc))
        got = dc.numpy()
        assert np.array_equal(got[:, :n], np.maximum(want + bias, 0))
        assert np.array_equal(got[:, n:], c0[:, n:])
    # rounding: a sum of k products, each addition rounding half an ulp
    a, b = (rng.standard_normal((r, k)).astype(np.float32) for r in (m, n))
    da, db, dc = up(a), up(b), up(np.zeros((m, n), np.float32))
    hip.check(L.lmp_k_gemm_f32(0, 1, m, n, k, da.ptr, k, db.ptr, k, dc.ptr, n, 0))
    err = np.abs(dc.numpy() - a.astype(np.float64) @ b.T.astype(np.float64))
    assert np.all(err <= (k + 2) * 2.0 ** -24 * (np.abs(a.astype(np.float64)) @ np.abs(b.T.astype(np.float64))))
