"""GPU parity at the sizes where the kernels' choice of path changes.

  * reductions: one launch (the last block folds) up to 256 first-pass blocks
    of 4096 elements, two launches above; several calls in a row, since the
    last block resets the arrival counter for the next call;
  * level 2: fewer rows than a vector, the 256-row waves and 1024-row blocks,
    and matrices whose columns are aligned (lda % 4 == 0) or not; the split of
    gemv's columns over a block's waves, and a triangle's runs that end inside
    a 1024-row chunk;
  * gemm: k-tiles shared by 2 or 4 groups of waves, with unequal shares.

References are numpy in float64 (whole-number data where the sums are exact in
either precision, so that those results compare exactly)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RNG_MAX = 7  # |entries| <= 7: sums of up to 1.5e5 products stay below 2^24


def _ints(rng, shape, dtype):
    return rng.integers(-RNG_MAX, RNG_MAX + 1, size=shape).astype(dtype)


@pytest.mark.parametrize("prefix,dtype", [("s", np.float32), ("d", np.float64)])
@pytest.mark.parametrize("n", [1, 4096, 4097, 100_003, 256 * 4096, 256 * 4096 + 1])
def test_reductions_each_side_of_the_fused_limit(ctx, prefix, dtype, n):
    rng = np.random.default_rng(n)
    x, y = _ints(rng, n, dtype), _ints(rng, n, dtype)
    x[n // 3] = 11  # the only largest entry
    # few nonzeros keep the float32 sums exact
    x[rng.random(n) < 0.9] = 0
    x[n // 3] = 11
    dx, dy, out = ctx.upload(x), ctx.upload(y), ctx.upload(np.zeros(1, dtype))
    x64, y64 = x.astype(np.float64), y.astype(np.float64)
    for _ in range(3):
        assert getattr(ctx, prefix + "dot")(n, dx, 1, dy, 1) == x64 @ y64
        assert getattr(ctx, prefix + "asum")(n, dx, 1) == np.abs(x64).sum()
        nrm = float(getattr(ctx, prefix + "nrm2")(n, dx, 1))
        # the sum of squares is exact; the root and its scaling round
        assert abs(nrm - np.sqrt(x64 @ x64)) <= 2 * np.finfo(dtype).eps * nrm
        assert getattr(ctx, "i" + prefix + "amax")(n, dx, 1) == n // 3
        getattr(ctx, prefix + "dot_dev")(n, dx, 1, dy, 1, out)
        assert out.to_host()[0] == x64 @ y64


def _triangle(A, uplo, unit=False):
    T = np.tril(A) if uplo == 1 else np.triu(A)
    if unit:
        np.fill_diagonal(T, 1.0)
    return T


@pytest.mark.parametrize("prefix,dtype", [("s", np.float32), ("d", np.float64)])
@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 1023, 1025, 2050, 3333])
@pytest.mark.parametrize("pad", [0, 3])
def test_level2_edges(ctx, prefix, dtype, n, pad):
    rng = np.random.default_rng(10 * n + pad)
    lda = n + pad
    A = _ints(rng, (n, lda), dtype)  # row j is column j
    x, y = _ints(rng, n, dtype), _ints(rng, n, dtype)
    M, x64, y64 = A[:, :n].T.astype(np.float64), x.astype(np.float64), y.astype(np.float64)
    nan = A.copy()
    dA, dx = ctx.upload(A), ctx.upload(x)
    for trans in (0, 1):
        dy = ctx.upload(y)
        getattr(ctx, prefix + "gemv")(trans, n, n, 2.0, dA, lda, dx, 1, -1.0, dy, 1)
        assert np.array_equal(dy.to_host(), 2.0 * ((M.T if trans else M) @ x64) - y64)
    for uplo in (1, 2):
        # NaN outside the triangle and in the padding: read at most, never used
        keep = np.zeros((n, lda), bool)
        keep[:, :n] = (np.tri(n) if uplo == 1 else np.tri(n).T).T
        nan = np.where(keep, A, np.nan).astype(dtype)
        dN = ctx.upload(nan)
        T = _triangle(M, uplo)
        S = T + T.T - np.diag(np.diag(M))
        dy = ctx.upload(y)
        getattr(ctx, prefix + "symv")(uplo, n, 2.0, dN, lda, dx, 1, -1.0, dy, 1)
        assert np.array_equal(dy.to_host(), 2.0 * (S @ x64) - y64)
        for trans in (0, 1):
            dy = ctx.upload(y)
            getattr(ctx, prefix + "trmv")(uplo, trans, 0, n, dN, lda, dx, 1, dy, 1)
            assert np.array_equal(dy.to_host(), (T.T if trans else T) @ x64)
        dy = ctx.upload(y)
        dU = ctx.upload(A)
        getattr(ctx, prefix + "syr2")(uplo, n, 2.0, dx, 1, dy, 1, dU, lda)
        xy = np.outer(x64, y64)
        want = A.astype(np.float64).copy()
        want[:, :n] = np.where(keep[:, :n], (M + 2.0 * (xy + xy.T)).T, want[:, :n])
        assert np.array_equal(dU.to_host().reshape(n, lda), want)
    dG = ctx.upload(A)
    getattr(ctx, prefix + "ger")(n, n, 2.0, dx, 1, ctx.upload(y), 1, dG, lda)
    want = A.astype(np.float64).copy()
    want[:, :n] += 2.0 * np.outer(y64, x64)
    assert np.array_equal(dG.to_host().reshape(n, lda), want)


@pytest.mark.parametrize("prefix,dtype", [("s", np.float32), ("d", np.float64)])
@pytest.mark.parametrize("m,n,lda", [(1024, 65536, 1024), (1027, 33001, 1027), (1027, 33001, 1028), (2050, 32770, 2052),
                                     (1279, 32765, 1280), (3, 66001, 3), (4097, 13003, 4097)])
def test_gemv_wide_blocks(ctx, prefix, dtype, m, n, lda):
    """1024-row blocks over many columns: whole waves, waves that cross m (by rows m % 4 and by whole lanes), fewer
    rows than a vector, columns that are no multiple of the step, each alignment."""
    rng = np.random.default_rng(m + n + lda)
    A = _ints(rng, (n, lda), np.int8)  # row j is column j; whole numbers, |sums| <= 49 n + 7 < 2^24
    x, y = _ints(rng, n, dtype), _ints(rng, m, dtype)
    x[rng.random(n) < 0.2] = 0
    dA, dx, dy = ctx.upload(A.astype(dtype)), ctx.upload(x), ctx.upload(y)
    try:
        getattr(ctx, prefix + "gemv")(0, m, n, 2.0, dA, lda, dx, 1, -1.0, dy, 1)
        want = 2.0 * (x.astype(np.float64) @ A[:, :m].astype(np.float64)) - y
        assert np.array_equal(dy.to_host(), want)
    finally:
        for buf in (dA, dx, dy):
            buf.free()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(1024, 1024, 256), (1000, 1025, 263), (1024, 1024, 545), (900, 1100, 1090),
                                   (1500, 1400, 301), (2048, 1024, 320)])
def test_sgemm_k_groups(ctx, ta, tb, m, n, k):
    """8 k-tiles of 32 and more: equal and unequal shares, a partial last k-tile, edge tiles. Exact: whole
    numbers, |sums| <= 49 k + 1 < 2^24."""
    rng = np.random.default_rng(m + n + k)
    A, B = _ints(rng, (m, k) if ta else (k, m), np.float32), _ints(rng, (k, n) if tb else (n, k), np.float32)
    C = _ints(rng, (n, m), np.float32)
    dC = ctx.upload(C)
    ctx.sgemm(ta, tb, m, n, k, 1.0, ctx.upload(A), k if ta else m, ctx.upload(B), n if tb else k, -1.0, dC, m)
    opA = A if ta else A.T  # m x k
    opB = B if tb else B.T  # k x n
    want = (opA.astype(np.float64) @ opB.astype(np.float64)).T - C
    assert np.array_equal(dC.to_host().reshape(n, m), want)
