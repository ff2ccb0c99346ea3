"""GPU parity at the sizes where the kernels' choice of path changes.

  * reductions: one launch (the last block folds) up to 256 first-pass blocks
    of 4096 elements, two launches above; several calls in a row, since the
    last block resets the arrival counter for the next call;
  * level 2: fewer rows than a vector, the 256-row waves and 1024-row blocks,
    and matrices whose columns are aligned (lda % 4 == 0) or not; the split of
    gemv's columns over a block's waves, and a triangle's runs that end inside
    a 1024-row chunk;
  * gemm: k-tiles shared by 2 or 4 groups of waves, with equal and unequal
    shares (the group count that the shapes are there for is checked on the CPU
    too, against the kernel that the library launches).

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
@pytest.mark.parametrize("n", [1, 3, 4, 5, 255, 257, 1023, 1025, 2050, 3333, 5125])
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


@pytest.mark.parametrize("prefix,dtype", [("s", np.float32), ("d", np.float64)])
@pytest.mark.parametrize("lda", [8192, 8195])
def test_gemv_sums_a_step_before_it_adds_it(ctx, prefix, dtype, lda):
    """A 1 followed by products that are each too small to change it: with u half an ulp of 1, one chain over the
    256 columns of the first split loses 255 * 0.99 u. A chain of 8 products a step (u each), an add for each of
    256 / 8 steps, one for each of the 32 splits and 8 for alpha, beta
    and the fold stay within 80 u of 1."""
    m = n = 8192
    u = np.finfo(dtype).eps / 2
    A = np.full((n, lda), 0.99 * u, dtype)
    A[0] = 1
    dA, dx, dy = ctx.upload(A), ctx.upload(np.ones(n, dtype)), ctx.upload(np.zeros(m, dtype))
    try:
        getattr(ctx, prefix + "gemv")(0, m, n, 1.0, dA, lda, dx, 1, 0.0, dy, 1)
        # differences from 1 are exact; what is wanted of them is (n - 1) products
        over = (dy.to_host() - dtype(1)).astype(np.float64)
        assert np.abs(over - (n - 1) * float(A[1, 0])).max() <= 80 * u
    finally:
        for buf in (dA, dx, dy):
            buf.free()


def _k_groups(m, n, k, uplo=0):
    """How many groups of waves share a 64 x 64 tile's k-tiles of 32 on 256 CUs."""
    tm, tn = -(-m // 64), -(-n // 64)
    assert not uplo or m == n
    tiles = tm * (tm + 1) // 2 if uplo else tm * tn
    ktiles = -(-k // 32)
    if tiles <= 256:
        return 4 if ktiles >= 64 else 2 if ktiles >= 16 else 1
    return 2 if tiles <= 512 and ktiles >= 64 else 1


# (m, n, k, padding of every leading dimension, groups)
K_GROUPS = [
    (1024, 1024, 545, 0, 2),  # 18 k-tiles, 9 each, whole tiles, a partial last k-tile
    (1000, 1001, 1040, 0, 2),  # 33: 17 and 16, edge tiles
    (1024, 900, 549, 4, 2),  # 18, an edge in n, a last k-tile of 5
    (640, 640, 2049, 0, 4),  # 65: 17 16 16 16, one column in the last k-tile
    (500, 700, 2113, 1, 4),  # 67: 17 17 17 16, edges, leading dimensions that are no multiple of 4
    (640, 640, 2112, 0, 4),  # 66: 17 17 16 16, whole k-tiles
    (640, 577, 2048, 64, 4),  # 64, equal shares
    (1500, 1000, 2081, 0, 2),  # 384 tiles, 66 k-tiles
    (1280, 1600, 2112, 1, 2),  # 500 tiles, 33 each
]
# just outside the rule: too few k-tiles, or more tiles than CUs
ONE_GROUP = [(1024, 1024, 256, 0, 1), (1000, 1025, 263, 0, 1), (900, 1100, 1090, 0, 1), (1500, 1400, 301, 0, 1),
             (2048, 1024, 320, 0, 1)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,pad,groups", K_GROUPS + ONE_GROUP)
def test_sgemm_k_groups(ctx, ta, tb, m, n, k, pad, groups):
    """Equal and unequal shares, edge tiles, partial last k-tiles, operands at any alignment. Exact: whole numbers,
    |sums| <= 49 k + 7 < 2^24."""
    assert _k_groups(m, n, k) == groups
    rng = np.random.default_rng(m + n + k)
    rows_a, rows_b = (k if ta else m) + pad, (n if tb else k) + pad
    A, B = _ints(rng, (m if ta else k, rows_a), np.float32), _ints(rng, (k if tb else n, rows_b), np.float32)
    C = _ints(rng, (n, m + pad), np.float32)
    dC = ctx.upload(C)
    ctx.sgemm(ta, tb, m, n, k, 1.0, ctx.upload(A), rows_a, ctx.upload(B), rows_b, -1.0, dC, m + pad)
    A, B = A[:, :k if ta else m], B[:, :n if tb else k]
    opA = A if ta else A.T  # m x k
    opB = B if tb else B.T  # k x n
    want = C.astype(np.float64)
    want[:, :m] = (opA.astype(np.float64) @ opB.astype(np.float64)).T - C[:, :m]
    assert np.array_equal(dC.to_host().reshape(n, m + pad), want)


@pytest.mark.parametrize("uplo", [1, 2])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("n,k,groups", [(1001, 1040, 2), (700, 2113, 4)])
def test_sgemmtr_k_groups(ctx, uplo, ta, tb, n, k, groups):
    """The same on a triangle's tiles; the other triangle is untouched."""
    assert _k_groups(n, n, k, uplo) == groups
    rng = np.random.default_rng(n + k)
    A, B = _ints(rng, (n, k) if ta else (k, n), np.float32), _ints(rng, (k, n) if tb else (n, k), np.float32)
    C = _ints(rng, (n, n), np.float32)
    dC = ctx.upload(C)
    ctx.sgemmtr(uplo, ta, tb, n, n, k, 1.0, ctx.upload(A), k if ta else n, ctx.upload(B), n if tb else k, -1.0, dC, n)
    opA, opB = (A if ta else A.T).astype(np.float64), (B if tb else B.T).astype(np.float64)
    keep = np.tri(n, dtype=bool) if uplo == 1 else np.tri(n, dtype=bool).T
    want = np.where(keep.T, (opA @ opB).T - C, C)
    assert np.array_equal(dC.to_host().reshape(n, n), want)
