"""The fp32 GEMM that runs on the bf16 matrix cores, each operand in three
parts (K > 32 and M > 32 with an operand transposed), through the C ABI, and
beside it the forward product X * W of the same shapes, which stays on the fp32
MFMAs: tile edges, K remainders, splits of K, unaligned rows, the whole range of
fp32, and values that are not finite."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # half an ulp of fp32, relative


def _run(hip, A, B, ta, tb, pad=(0, 0), c0=None, acc=0, colsum=False):
    """C = op(A) op(B) with `pad` extra values in each stored row (poisoned)
    and C's rows; the column sums of op(B) beside it when asked for."""
    m, k = A.shape[::-1] if ta else A.shape
    n = B.shape[0] if tb else B.shape[1]
    bufs = []
    for x, p in ((A, pad[0]), (B, pad[1])):
        y = np.full((x.shape[0], x.shape[1] + p), np.nan, np.float32)
        y[:, :x.shape[1]] = x
        bufs.append((hip.DeviceBuffer.from_numpy(y), y.shape[1]))
    ldc = n + pad[1]
    c = np.full((m, ldc), 7.0, np.float32)
    if c0 is not None:
        c[:, :n] = c0
    dc = hip.DeviceBuffer.from_numpy(c)
    (da, lda), (db, ldb) = bufs
    if colsum:
        cs = hip.DeviceBuffer.from_numpy(np.full(n, 3.0, np.float32))
        hip.check(hip.lib().lmp_k_gemm_colsum_f32(ta, tb, m, n, k, da.ptr, lda, db.ptr, ldb,
                                                  dc.ptr, ldc, acc, cs.ptr, 0))
        got = dc.numpy()
        assert np.all(got[:, n:] == 7.0)
        return got[:, :n], cs.numpy()
    hip.check(hip.lib().lmp_k_gemm_f32(ta, tb, m, n, k, da.ptr, lda, db.ptr, ldb, dc.ptr, ldc, acc))
    got = dc.numpy()
    assert np.all(got[:, n:] == 7.0)  # nothing outside C
    return got[:, :n]


def _operands(m, n, k, ta, tb, seed):
    rng = np.random.default_rng(seed)
    a = rng.standard_normal((m, k), dtype=np.float32)
    b = rng.standard_normal((k, n), dtype=np.float32)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    return (np.ascontiguousarray(a.T) if ta else a), (np.ascontiguousarray(b.T) if tb else b), a64, b64


# Tile edges of the five tile sizes, K around one, two and three steps of 16
# and around the ends of K splits; the last five take the 256 x 256, 256 x 128,
# 128 x 128, 64 x 128 and 64 x 64 tiles.
SHAPES = [(33, 1, 33), (64, 65, 47), (65, 64, 48), (129, 127, 49), (257, 255, 63), (255, 130, 64),
          (40, 1000, 1003), (200, 200, 2049), (4096, 4000, 49), (512, 2050, 2083), (1000, 1027, 1531),
          (64, 2048, 1030), (300, 700, 260)]


@pytest.mark.parametrize("m,n,k", SHAPES, ids=str)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_against_float64(hip, m, n, k, ta, tb):
    """Rounding errors only: a step of 16 k adds six bf16 products, each with
    at most two roundings of half an ulp of the running sum, independent of
    each other, so the 2-norm of the error is below sqrt(12 ceil(K / 16))
    half-ulps of the result's (a missing part of a split, 2^-17 of a term, is
    over it).  Aligned and odd row pitches give the same bits."""
    if not ta and not tb:
        m += 512  # the fp32 MFMAs, within the same bounds
    A, B, a64, b64 = _operands(m, n, k, ta, tb, m * 31 + n * 7 + k)
    want = a64 @ b64
    got = _run(hip, A, B, ta, tb)
    steps = -(-k // 16)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err <= np.sqrt(12 * steps + 2) * U, err
    # every element, against the terms' magnitudes
    assert np.all(np.abs(got - want) <= (12 * steps + 70) * U * (np.abs(a64) @ np.abs(b64)))
    padded = _run(hip, A, B, ta, tb, pad=(1, 3))
    assert np.array_equal(padded.view(np.uint32), got.view(np.uint32))
    c0 = np.random.default_rng(1).standard_normal((m, n), dtype=np.float32)
    acc = _run(hip, A, B, ta, tb, pad=(3, 1), c0=c0, acc=1)
    assert np.array_equal(acc.view(np.uint32), (c0 + got).view(np.uint32))


# K just above 32 and long, on tiles whose leading products accumulate apart, and
# (last) the 256 x 256 tile's one sum.
@pytest.mark.parametrize("m,n,k", [(200, 256, 33), (512, 512, 40), (2048, 2048, 2048), (4096, 4096, 65)], ids=str)
@pytest.mark.parametrize("family", ["normal", "dominated", "spread", "constant", "single"])
def test_error_by_operand_family(hip, family, m, n, k):
    """Operands besides normal ones: one term of each row 2^12 times the others,
    terms spread over 2^40, equal terms whose parts left out have one sign, and a
    single product per element.

    The running sum is rounded once per 16 k (six times in the one sum), each
    rounding at most an ulp and 0.58 half-ulps rms; averaged over a walk that
    starts at zero and over mantissas 0.41 sqrt(roundings) half-ulps of the
    result, 0.6 with the margin.  A single product is one addition: half an ulp,
    half of one for the parts left out, and in the one sum, where it is the last
    of six, up to another for the alignment of the smaller summand."""
    rng = np.random.default_rng(m + k)
    big = m * n >= 1 << 24
    a, b = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n)))
    if family == "dominated":
        a[np.arange(m), rng.integers(0, k, m)] *= np.float32(4096)
    elif family == "spread":
        a *= np.exp2(rng.uniform(-20, 20, (m, k))).astype(np.float32)
    elif family == "constant":
        a[:], b[:] = np.float32(1 + 2.0 ** -8 - 2.0 ** -17), np.float32(1 + 2.0 ** -8 - 2.0 ** -17)
    elif family == "single":
        a = rng.random((m, k), dtype=np.float32) + 1
        b = np.zeros((k, n), np.float32)
        b[np.arange(n) % k, np.arange(n)] = rng.random(n, dtype=np.float32) + 1
    want = a[:512].astype(np.float64) @ b.astype(np.float64)
    got = _run(hip, np.ascontiguousarray(a.T), b, 1, 0)[:512]
    err = np.abs(got - want)
    roundings = -(-k // 16) * (6 if big else 1)
    if family == "single":
        assert np.max(err / np.abs(want)) <= (3 if big else 2) * U * (1 + 2.0 ** -6)
    elif family == "constant":  # every rounding may have one sign
        assert np.max(err / np.abs(want)) <= (2 * roundings + 2) * U
    else:
        assert np.linalg.norm(err) <= (0.6 * np.sqrt(roundings) + 1) * U * np.linalg.norm(want)


@pytest.mark.parametrize("m,n,k", [(129, 127, 49), (1000, 1027, 1531), (200, 200, 2049), (300, 700, 260)],
                         ids=str)
def test_column_sums(hip, m, n, k):
    """The column sums beside the product (whole and split K, odd pitches):
    within K half-ulps of the terms' magnitudes, the product unchanged."""
    A, B, a64, b64 = _operands(m, n, k, 1, 0, 11)
    for pad in ((0, 0), (1, 3)):
        got, cs = _run(hip, A, B, 1, 0, pad=pad, colsum=True)
        assert np.array_equal(got.view(np.uint32), _run(hip, A, B, 1, 0).view(np.uint32))
        assert np.all(np.abs(cs - b64.sum(0)) <= k * U * np.abs(b64).sum(0))


@pytest.mark.parametrize("m,k", [(64, 64), (200, 96), (300, 256)], ids=str)
@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 1), (1, 0)])
def test_every_finite_value_survives(hip, m, k, ta, tb):
    """Random bit patterns of finite fp32 values, subnormals and the largest
    included, times the identity (its own transpose): each row exactly, through
    either operand."""
    rng = np.random.default_rng(m + k)
    bits = rng.integers(0, 1 << 32, (m, k), dtype=np.uint64).astype(np.uint32)
    bits[(bits & 0x7f800000) == 0x7f800000] ^= 0x00800000  # no infinity, no NaN
    bits[::3] &= np.uint32(0x807fffff)                      # whole rows of subnormals
    x = bits.view(np.float32)
    x = np.where(x == 0, np.float32(1e-45), x)
    eye = np.eye(k, dtype=np.float32)
    got = _run(hip, np.ascontiguousarray(x.T) if ta else x, eye, ta, tb)
    assert np.array_equal(got.view(np.uint32), x.view(np.uint32))
    y = np.ascontiguousarray(x.T)  # [k, m]
    got = _run(hip, eye, np.ascontiguousarray(y.T) if tb else y, ta, tb)
    assert np.array_equal(got.view(np.uint32), y.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(40, 70, 40), (300, 270, 200), (200, 200, 2049)], ids=str)
@pytest.mark.parametrize("kind", ["inf", "nan", "large", "overflow"])
def test_values_that_are_not_finite(hip, m, n, k, kind):
    """One infinity, NaN, row near the top of the range, or row whose results
    overflow, alone in its tile: C is as float64 has it (rounded to fp32)."""
    A, B, _, _ = _operands(m, n, k, 0, 0, 5)
    row = m - 3
    if kind == "inf":
        A[row, 1] = np.inf
    elif kind == "nan":
        A[row, 1] = np.nan
    elif kind == "large":
        A[row] *= np.float32(1e33)
    else:
        A[row] = (np.abs(A[row]) + 1) * np.float32(1e37)
        B[:, 2] = np.abs(B[:, 2]) + 1
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
        want32 = want.astype(np.float32)
    got = _run(hip, np.ascontiguousarray(A.T), B, 1, 0)
    if kind == "overflow":  # the other columns' terms overflow one by one, with either sign
        keep = np.ones((m, n), bool)
        keep[row] = False
        keep[row, 2] = True
    else:
        keep = np.ones((m, n), bool)
    assert np.array_equal(np.isnan(got)[keep], np.isnan(want32)[keep])
    inf = np.isinf(want32) & keep
    assert np.array_equal(got[inf], want32[inf])
    fin = np.isfinite(want32) & keep
    scale = np.abs(np.where(np.isfinite(A), A, 0)).astype(np.float64) @ np.abs(B).astype(np.float64)
    # the fallback's fp32 products round once per value of k
    assert np.all(np.abs(got[fin] - want[fin]) <= (2 * k + 70) * U * scale[fin])


@pytest.mark.parametrize("n,k", [(256, 64), (1000, 160), (77, 333)], ids=str)
def test_forward_rows_keep_their_bits(hip, n, k):
    """X * W rounds the same whatever its number of rows (sizes with one tile and
    no split of K): the first rows of a longer batch are the shorter one's."""
    A, B, _, _ = _operands(1600, n, k, 0, 0, n)
    want = _run(hip, A[:512], B, 0, 0)
    for m in (513, 640, 1600):
        assert np.array_equal(_run(hip, A[:m], B, 0, 0)[:512].view(np.uint32), want.view(np.uint32)), m


@pytest.mark.parametrize("m,n,k", [(300, 270, 200), (200, 200, 2049), (260, 130, 37), (1100, 1100, 50)], ids=str)
@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0), (1, 1)])
def test_tiles_computed_again(hip, m, n, k, ta, tb):
    """Rows near the top of the range send every tile to the fp32 products, in
    each orientation, with K tails, short splits and odd pitches: within their
    rounding (one per value of k) everywhere, C's other columns untouched."""
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    a[::29] *= np.float32(1e33)
    want = a.astype(np.float64) @ b.astype(np.float64)
    scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
    A, B = (np.ascontiguousarray(a.T) if ta else a), (np.ascontiguousarray(b.T) if tb else b)
    got = _run(hip, A, B, ta, tb)
    assert np.all(np.abs(got - want) <= (k + 70) * U * scale)
    assert np.array_equal(_run(hip, A, B, ta, tb, pad=(1, 3)).view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("m,n,k", [(2048, 2048, 2048), (1024, 1027, 4096), (700, 900, 100), (300, 511, 257)], ids=str)
@pytest.mark.parametrize("positive", [False, True], ids=["normal", "positive"])
def test_column_sums_close_to_float64(hip, m, n, k, positive):
    """The column sums, whole K and split: a step's 4 or 8 values add in up to
    three levels, the steps' and splits' errors are kept, and up to four parts
    meet, so eight independent roundings of 0.58 half-ulps rms at most, whatever
    K is (a quarter more for the sample)."""
    A, B, _, b64 = _operands(m, n, k, 1, 0, n)
    if positive:
        B, b64 = np.abs(B), np.abs(b64)
    want = b64.sum(0)
    for pad in ((0, 0), (1, 3)):
        _, cs = _run(hip, A, B, 1, 0, pad=pad, colsum=True)
        assert np.linalg.norm(cs - want) <= 1.25 * 0.58 * np.sqrt(8) * U * np.linalg.norm(want)


@pytest.mark.parametrize("k", [100, 2049])
def test_column_sums_that_are_not_finite(hip, k):
    """Infinities and NaN in a column, sums that overflow, columns of the largest
    magnitudes that cancel: as the plain sum has them."""
    m, n = 200, 70
    A, B, _, _ = _operands(m, n, k, 1, 0, 3)
    big = np.float32(3e38)
    B[k // 2, 3], B[k // 3, 4], B[5, 5], B[7, 6], B[9, 6] = np.inf, -np.inf, np.nan, np.inf, -np.inf
    B[:, 8] = big
    B[:, 9] = 0
    B[[20, 90], 9] = big, -big
    _, cs = _run(hip, A, B, 1, 0, colsum=True)
    assert cs[3] == np.inf and cs[4] == -np.inf and np.isnan(cs[5]) and np.isnan(cs[6])
    assert cs[8] == np.inf and cs[9] == 0
    ok = np.ones(n, bool)
    ok[[3, 4, 5, 6, 8]] = False
    assert np.all(np.isfinite(cs[ok]))
