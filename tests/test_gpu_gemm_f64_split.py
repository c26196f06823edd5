"""float64 GEMM on 64 x 64 tiles with K split: tile edges, K remainders and
the ends of splits, every orientation, aligned and odd rows, accumulate."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# K of one to three tiles of 16 and a remainder, splits with a short last part,
# few and many tiles of C, as many as the CUs.
SHAPES = [(1, 1, 1), (64, 64, 15), (65, 63, 16), (64, 128, 33), (33, 130, 48), (32, 32, 2048), (96, 96, 2047),
          (200, 200, 2001), (700, 70, 129), (1030, 1020, 70)]


@pytest.mark.parametrize("m,n,k", SHAPES, ids=str)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_gemm_f64_split(hip, m, n, k, ta, tb):
    rng = np.random.default_rng(m + n + k)
    L = hip.lib()
    for pad in (0, 1):
        # small integers: every sum is exact in any order
        a = rng.integers(-8, 9, (m, k)).astype(np.float64)
        b = rng.integers(-8, 9, (k, n)).astype(np.float64)
        c0 = rng.integers(-8, 9, (m, n)).astype(np.float64)
        want = a @ b

        def up(x, t):
            x = x.T if t else x
            y = np.full((x.shape[0], x.shape[1] + pad), np.nan)
            y[:, :x.shape[1]] = x
            return hip.DeviceBuffer.from_numpy(y), y.shape[1]

        (da, lda), (db, ldb), (dc, ldc) = up(a, ta), up(b, tb), up(c0, 0)
        for acc in (1, 0):
            hip.check(L.lmp_k_gemm(hip.FLOAT64, ta, tb, m, n, k, da.ptr, lda, db.ptr, ldb, dc.ptr, ldc, acc))
            got = dc.numpy()
            assert np.array_equal(got[:, :n], c0 + want if acc else want), (pad, acc)
            assert np.all(np.isnan(got[:, n:]))
    # rounding: a sum of k products, each rounding half an ulp of the terms
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    (da, lda), (db, ldb), (dc, ldc) = up(a, ta), up(b, tb), up(c0, 0)
    hip.check(L.lmp_k_gemm(hip.FLOAT64, ta, tb, m, n, k, da.ptr, lda, db.ptr, ldb, dc.ptr, ldc, 0))
    err = np.abs(dc.numpy()[:, :n] - a @ b)
    assert np.all(err <= 2 * k * 2.0 ** -53 * (np.abs(a) @ np.abs(b)))
