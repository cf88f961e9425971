"""f32 matmul with f64 accumulation (matmul, matmul_bias, matmul_strided_batched;
mod.rs:54-86, 561-591) at the edges of its kernels: 1-4 rows (row and column
streams, their k splits and ragged widths), the 32 and 64 tiles, k tails of a
32-value step, k splits, and every transpose.  f32 products are exact in f64,
so a result differs from the f64 reference by its one rounding (2^-24) and the
order of f64 additions (k 2^-53 of the sum of magnitudes, far below it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
F = np.float32

SHAPES = [  # batch, m, k, n
    (1, 1, 1, 1), (2, 1, 129, 77), (32, 1, 101, 128), (1, 2, 1001, 12), (3, 3, 33, 70), (1, 4, 4100, 260),
    (1, 1, 2048, 4100), (1, 5, 3, 7), (2, 33, 31, 65), (3, 17, 100, 129), (1, 37, 128, 37), (1, 200, 768, 50),
    (1, 65, 2052, 68), (1, 70, 4097, 66), (2, 70, 33, 66), (12, 64, 64, 64), (1, 1030, 70, 1029),
]


def _check(c, a, b, extra=0.0):
    ref = np.matmul(a.astype(np.float64), b.astype(np.float64)) + extra
    mag = np.matmul(np.abs(a).astype(np.float64), np.abs(b).astype(np.float64)) + np.abs(extra)
    bound = 2.0 ** -23 * np.abs(ref) + a.shape[-1] * 2.0 ** -52 * mag
    assert (np.abs(c.astype(np.float64) - ref) <= bound).all()


@pytest.mark.parametrize("bt,m,k,n", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_matmul_f64_accumulation(hip, bt, m, k, n, ta, tb):
    print(f"[case] {bt} x {m} x {k} x {n} ta={ta} tb={tb}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m * k + n + bt)
    a = rng.normal(size=(bt, m, k)).astype(F)
    b = rng.normal(size=(bt, k, n)).astype(F)
    A = B.from_vec(np.ascontiguousarray(a.swapaxes(1, 2) if ta else a))
    W = B.from_vec(np.ascontiguousarray(b.swapaxes(1, 2) if tb else b))
    c = B.matmul_strided_batched(A, W, bt, m, k, n, bool(ta), bool(tb)).to_vec().reshape(bt, m, n)
    _check(c, a, b)
    if bt == 1:
        bias = rng.normal(size=n).astype(F)
        plain = B.matmul(A, W, m, k, n, bool(ta), bool(tb)).to_vec()
        assert np.array_equal(plain, c.ravel())
        got = B.matmul_bias(A, W, B.from_vec(bias), m, k, n, bool(ta), bool(tb)).to_vec()
        assert np.array_equal(got, (plain.reshape(m, n) + bias).ravel())  # the rounded product, then an f32 add


@pytest.mark.parametrize("m", [1, 3, 40])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_matmul_nonfinite_stays_in_its_rows_and_columns(hip, m, ta, tb):
    """Padding must not turn an infinity into a NaN elsewhere."""
    print(f"[case] m={m} ta={ta} tb={tb}", flush=True)
    B = hip.HipBackend
    k, n = 37, 45
    rng = np.random.default_rng(m)
    a = np.abs(rng.normal(size=(m, k))).astype(F) + F(0.1)
    b = np.abs(rng.normal(size=(k, n))).astype(F) + F(0.1)
    a[m // 2, 5] = np.inf
    b[7, n - 1] = np.nan
    c = B.matmul(B.from_vec(np.ascontiguousarray(a.T if ta else a)), B.from_vec(np.ascontiguousarray(b.T if tb else b)),
                 m, k, n, bool(ta), bool(tb)).to_vec().reshape(m, n)
    with np.errstate(invalid="ignore"):
        ref = (a.astype(np.float64) @ b.astype(np.float64)).astype(F)
    assert np.array_equal(np.isnan(c), np.isnan(ref)) and np.array_equal(np.isinf(c), np.isinf(ref))


def _block_bytes(n):
    """The pool's size class of an n-byte storage: (8 + i) << (e + 5) bytes."""
    return next(c for e in range(40) for c in ((8 + i) << (e + 5) for i in range(8)) if c >= n)


@pytest.mark.parametrize("k", [33, 34, 35, 65, 4097])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_matmul_reads_nothing_past_a_matrix(hip, k, ta, tb):
    """What lies behind the k tail of an operand - the next batch entry, and
    after the last entry the rest of its storage block - is NaN: no product may
    take it up (a tail position times a stale NaN would show)."""
    print(f"[case] k={k} ta={ta} tb={tb}", flush=True)
    B = hip.HipBackend
    bt, m, n = 3, 70, 66
    rng = np.random.default_rng(k + 2 * ta + tb)
    a = rng.normal(size=(bt, m, k)).astype(F)
    b = rng.normal(size=(bt, k, n)).astype(F)
    a[1] = np.nan  # entry 0 borders on it, entry 2 on the rest of the block
    b[1] = np.nan

    def storage(x):  # in a block that was all NaN before
        B.from_vec(np.full(_block_bytes(x.nbytes) // 4, np.nan, F)).free()
        return B.from_vec(np.ascontiguousarray(x))

    A, W = storage(a.swapaxes(1, 2) if ta else a), storage(b.swapaxes(1, 2) if tb else b)
    c = B.matmul_strided_batched(A, W, bt, m, k, n, bool(ta), bool(tb)).to_vec().reshape(bt, m, n)
    assert np.isnan(c[1]).all()
    _check(c[::2], a[::2], b[::2])


TOP = 2 ** 31 - 1  # the largest dimension an entry point takes


@pytest.mark.parametrize("m,k,n,tb", [(1, TOP, 1, 1), (1, TOP - 1024, 1, 0), (5, TOP, 1, 1), (TOP, 1, 1, 0),
                                     (1, 1, TOP, 0), (TOP - 1024, 1, 1, 0)])
def test_matmul_largest_dimension(hip, m, k, n, tb):
    """A dimension whose last tile or stride ends past 2^31 - 1.  Products of
    ones: the f64 sums are exact, so a position left out or taken twice shows."""
    print(f"[case] {m} x {k} x {n} tb={tb}", flush=True)
    B = hip.HipBackend
    c = B.matmul(B.ones(m * k), B.ones(k * n), m, k, n, False, bool(tb))
    if m * n < 100:
        assert (c.to_vec() == F(k)).all()
    else:
        assert c.n == m * n and B.sum(c) == F(m * n)


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,k,n", [(5, 33, 2 ** 21 + 41), (2 ** 21 + 41, 33, 5), (6, 2 ** 21 + 41, 7)])
def test_matmul_wide(hip, m, k, n, ta, tb):
    """A dimension above 2^21: loads with 64-bit addresses."""
    print(f"[case] {m} x {k} x {n} ta={ta} tb={tb}", flush=True)
    B = hip.HipBackend
    rng = np.random.default_rng(m + k + n)
    a = rng.normal(size=(1, m, k)).astype(F)
    b = rng.normal(size=(1, k, n)).astype(F)
    A = B.from_vec(np.ascontiguousarray(a.swapaxes(1, 2) if ta else a))
    W = B.from_vec(np.ascontiguousarray(b.swapaxes(1, 2) if tb else b))
    _check(B.matmul(A, W, m, k, n, bool(ta), bool(tb)).to_vec().reshape(1, m, n), a, b)


def test_matmul_more_tiles_than_workgroups(hip):
    """2^22 + 9 batch entries: a workgroup takes several tiles."""
    B = hip.HipBackend
    bt, m, k, n = 2 ** 22 + 9, 2, 3, 2
    rng = np.random.default_rng(5)
    a = rng.normal(size=(bt, m, k)).astype(F)
    b = rng.normal(size=(bt, k, n)).astype(F)
    _check(B.matmul_strided_batched(B.from_vec(a), B.from_vec(b), bt, m, k, n).to_vec().reshape(bt, m, n), a, b)
