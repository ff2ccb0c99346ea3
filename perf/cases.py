"""Timed calls of the library's public entry points (wgblas_amd.Context) on GPU-resident operands.

A case is one routine of the BLAS at one size, precision and set of options:

  * level 1: a vector's four reductions (dot, asum, nrm2, iamax), with the
    results on the host (the default of the JavaScript API) or left in
    device memory (a solver that goes on on the GPU);
  * level 2: gemv, ger, symv, trmv, syr2;
  * level 3: gemm, gemmtr, syrk, syr2k, symm, trmm, trsm.

`listed()` holds the sizes of the repository's own benchmark (sgemm 512,
sgemm 8192, the ragged 8191 x 8193 x 4097, dgemm 4096, ssyrk 8192 / 4096,
strsm 4096, reductions at 2^28, ssymv at 16384) beside ordinary smaller ones
(sgemm 1024, sgemv 4096, reductions of 100 003 elements, ssyr2 at 8191);
`draw()` gives the same routines over the whole range of sizes, both
precisions, every transpose / triangle / side option and padded leading
dimensions.

Matrices are column-major; a rows x cols matrix is kept as a torch tensor of
shape (cols, ld), whose row j is column j.
"""
import math

import torch

import wgblas_amd as wg

F32, F64 = "f32", "f64"
TORCH = {F32: torch.float32, F64: torch.float64}
SIZE = {F32: 4, F64: 8}
EPS = {F32: 2.0 ** -24, F64: 2.0 ** -53}

_ctx = None


def _context():
    """The device handle that a program opens once and keeps."""
    global _ctx
    if _ctx is None:
        _ctx = wg.Context(0)
    return _ctx


# ---- the cases -----------------------------------------------------------------


def listed():
    return [
        # The scalar results of a short vector: what a solver's inner products cost when the
        # host waits for each of them; latency, launches and the copy back count.
        {"name": "reductions_100k_host", "op": "reductions", "t": F32, "n": 100_003, "inc": 1, "host": True},
        # The benchmark's vectors of 2^28 normals: the stream from HBM counts.
        {"name": "reductions_2e28", "op": "reductions", "t": F32, "n": 1 << 28, "inc": 1, "host": False},
        # A dense layer's or an iteration's matrix-vector product at an ordinary size.
        {"name": "sgemv_4096", "op": "gemv", "t": F32, "m": 4096, "n": 4096, "trans": 0, "pad": 0},
        # The benchmark's symmetric product: one triangle read once.
        {"name": "ssymv_16384", "op": "symv", "t": F32, "n": 16384, "uplo": 1, "pad": 0},
        # A rank-2 update of a triangle (tridiagonalisation, BFGS) at an odd order.
        {"name": "ssyr2_8191", "op": "syr2", "t": F32, "n": 8191, "uplo": 2, "pad": 2},
        # The benchmark's small product.
        {"name": "sgemm_512", "op": "gemm", "t": F32, "m": 512, "n": 512, "k": 512, "ta": 0, "tb": 0, "pad": 0, "beta": 0.0},
        # An ordinary product (the top of the reference's own benchmark sizes).
        {"name": "sgemm_1024", "op": "gemm", "t": F32, "m": 1024, "n": 1024, "k": 1024, "ta": 0, "tb": 1, "pad": 0, "beta": 0.0},
        # The benchmark's ragged product: edge tiles in every direction, leading dimensions of 1 mod 64.
        {"name": "sgemm_ragged", "op": "gemm", "t": F32, "m": 8191, "n": 8193, "k": 4097, "ta": 1, "tb": 0, "pad": 64, "beta": 0.5},
        # The benchmark's headline product.
        {"name": "sgemm_8192", "op": "gemm", "t": F32, "m": 8192, "n": 8192, "k": 8192, "ta": 0, "tb": 0, "pad": 0, "beta": 0.5},
        # The benchmark's double-precision product.
        {"name": "dgemm_4096", "op": "gemm", "t": F64, "m": 4096, "n": 4096, "k": 4096, "ta": 0, "tb": 1, "pad": 0, "beta": 1.0},
        # The benchmark's covariance-like update of one triangle.
        {"name": "ssyrk_8192", "op": "syrk", "t": F32, "n": 8192, "k": 4096, "uplo": 1, "trans": 0, "pad": 0},
        # The benchmark's triangular solve with many right-hand sides.
        {"name": "strsm_4096", "op": "trsm", "t": F32, "m": 4096, "n": 4096, "side": 1, "uplo": 1, "trans": 0, "diag": 0, "pad": 0},
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm; half of them rounded to multiples of 64 where that fits."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 0.5 and v >= 128:
        v = v // 64 * 64
    return max(lo, min(hi, v))


def draw(rng):
    op = rng.choice(["reductions", "gemv", "ger", "symv", "trmv", "syr2", "gemm", "gemm", "gemm", "gemm",
                     "gemmtr", "syrk", "syr2k", "symm", "trmm", "trsm"])
    t = F32 if op == "trsm" else rng.choice([F32, F32, F64])
    c = {"op": op, "t": t}
    if op == "reductions":
        inc = rng.choice([1, 1, 1, 3])
        c.update(n=_log(rng, 10_000, (1 << 26 if inc == 3 else 1 << 28) // (1 if t == F32 else 2)), inc=inc,
                 host=rng.random() < 0.5)
        return c
    c["pad"] = rng.choice([0, 0, 1, 4, 33])
    if op in ("gemv", "ger"):
        c.update(m=_log(rng, 512, 16384), n=_log(rng, 512, 16384))
        if op == "gemv":
            c["trans"] = rng.randrange(2)
    elif op in ("symv", "trmv", "syr2"):
        c.update(n=_log(rng, 512, 16384), uplo=rng.choice([1, 2]))
        if op == "trmv":
            c.update(trans=rng.randrange(2), diag=rng.randrange(2))
    elif op == "gemm":
        top = 8192 if t == F32 else 4096
        c.update(m=_log(rng, 256, top), n=_log(rng, 256, top), k=_log(rng, 256, top), ta=rng.randrange(2),
                 tb=rng.randrange(2), beta=rng.choice([0.0, 0.5]))
    elif op in ("gemmtr", "syrk", "syr2k"):
        top = 8192 if t == F32 else 4096
        c.update(n=_log(rng, 512, top), k=_log(rng, 256, 4096), uplo=rng.choice([1, 2]), trans=rng.randrange(2))
    else:
        c.update(m=_log(rng, 256, 4096), n=_log(rng, 256, 4096), side=rng.choice([1, 2]), uplo=rng.choice([1, 2]))
        if op != "symm":
            c.update(trans=rng.randrange(2), diag=rng.randrange(2))
    return c


# ---- inputs ----------------------------------------------------------------------


def _inputs(c, seed):
    """The operands, on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    dt = TORCH[c["t"]]

    def uniform(cols, rows, scale=1.0):
        # rows + pad is the leading dimension
        return torch.empty(cols, rows + c["pad"], dtype=dt, device="cuda").uniform_(-scale, scale, generator=g)

    def vector(n):
        return torch.empty(n, dtype=dt, device="cuda").uniform_(-1.0, 1.0, generator=g)

    op = c["op"]
    if op == "reductions":
        span = (c["n"] - 1) * c["inc"] + 1
        x = torch.empty(span, dtype=dt, device="cuda").normal_(generator=g)
        # correlated, as a solver's inner products are, so that the sum does not cancel
        y = torch.empty(span, dtype=dt, device="cuda").normal_(generator=g).add_(x, alpha=0.5)
        return {"x": x, "y": y}
    if op == "gemv":
        m, n = c["m"], c["n"]
        return {"A": uniform(n, m), "x": vector(m if c["trans"] else n), "y": vector(n if c["trans"] else m)}
    if op == "ger":
        return {"A": uniform(c["n"], c["m"]), "x": vector(c["m"]), "y": vector(c["n"])}
    if op in ("symv", "trmv", "syr2"):
        return {"A": uniform(c["n"], c["n"]), "x": vector(c["n"]), "y": vector(c["n"])}
    if op == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"A": uniform(m, k) if c["ta"] else uniform(k, m), "B": uniform(k, n) if c["tb"] else uniform(n, k),
                "C": uniform(n, m)}
    if op in ("gemmtr", "syrk", "syr2k"):
        n, k = c["n"], c["k"]
        d = {"A": uniform(n, k) if c["trans"] else uniform(k, n), "C": uniform(n, n)}
        if op != "syrk":
            d["B"] = uniform(n, k) if c["trans"] else uniform(k, n)
        return d
    order = c["m"] if c["side"] == wg.LEFT else c["n"]
    if op == "trsm":
        # well conditioned: off-diagonals in [-1/order, 1/order), diagonal 2
        A = uniform(order, order, 1.0 / order)
        A[:, :order].diagonal().fill_(2.0)
    else:
        A = uniform(order, order)
    d = {"A": A, "B": uniform(c["n"], c["m"])}
    if op == "symm":
        d["C"] = uniform(c["n"], c["m"])
    return d


def prepare(c, seed):
    s = {"case": dict(c), "ctx": _context()}
    s.update(_inputs(c, seed))
    if c["op"] == "reductions":
        s["out"] = torch.zeros(3, dtype=TORCH[c["t"]], device="cuda")
        s["index"] = torch.zeros(1, dtype=torch.int64, device="cuda")
    if c["op"] in ("trmm", "trsm"):
        s["X"] = torch.empty_like(s["B"])  # the right-hand sides stay; the product / solution goes here
    torch.cuda.synchronize()  # the handle's stream does not wait for torch's
    return s


# ---- one pass ----------------------------------------------------------------------


def _ptr(t):
    return t.data_ptr()


def run(s):
    c, ctx = s["case"], s["ctx"]
    return _RUN[c["op"]](s, c, ctx, "s" if c["t"] == F32 else "d")


def _reductions(s, c, ctx, p):
    n, inc, x, y = c["n"], c["inc"], _ptr(s["x"]), _ptr(s["y"])
    dot, asum, nrm2 = p + "dot", p + "asum", p + "nrm2"
    iamax = "i" + p + "amax"
    if c["host"]:
        return {"dot": float(getattr(ctx, dot)(n, x, inc, y, inc)), "asum": float(getattr(ctx, asum)(n, x, inc)),
                "nrm2": float(getattr(ctx, nrm2)(n, x, inc)), "index": int(getattr(ctx, iamax)(n, x, inc))}
    out, size = _ptr(s["out"]), SIZE[c["t"]]
    getattr(ctx, dot + "_dev")(n, x, inc, y, inc, out)
    getattr(ctx, asum + "_dev")(n, x, inc, out + size)
    getattr(ctx, nrm2 + "_dev")(n, x, inc, out + 2 * size)
    getattr(ctx, iamax + "_dev")(n, x, inc, _ptr(s["index"]))
    return {"sums": s["out"], "index": s["index"]}


def _gemv(s, c, ctx, p):
    m, n = c["m"], c["n"]
    getattr(ctx, p + "gemv")(c["trans"], m, n, 1.5, _ptr(s["A"]), m + c["pad"], _ptr(s["x"]), 1, 0.5, _ptr(s["y"]), 1)
    return s["y"]


def _ger(s, c, ctx, p):
    m, n = c["m"], c["n"]
    getattr(ctx, p + "ger")(m, n, 0.75, _ptr(s["x"]), 1, _ptr(s["y"]), 1, _ptr(s["A"]), m + c["pad"])
    return s["A"][:, :m]


def _symv(s, c, ctx, p):
    n = c["n"]
    getattr(ctx, p + "symv")(c["uplo"], n, 1.5, _ptr(s["A"]), n + c["pad"], _ptr(s["x"]), 1, 0.5, _ptr(s["y"]), 1)
    return s["y"]


def _trmv(s, c, ctx, p):
    n = c["n"]
    getattr(ctx, p + "trmv")(c["uplo"], c["trans"], c["diag"], n, _ptr(s["A"]), n + c["pad"], _ptr(s["x"]), 1, _ptr(s["y"]), 1)
    return s["y"]


def _syr2(s, c, ctx, p):
    n = c["n"]
    getattr(ctx, p + "syr2")(c["uplo"], n, 0.75, _ptr(s["x"]), 1, _ptr(s["y"]), 1, _ptr(s["A"]), n + c["pad"])
    return s["A"][:, :n]


def _gemm(s, c, ctx, p):
    m, n, k, pad = c["m"], c["n"], c["k"], c["pad"]
    getattr(ctx, p + "gemm")(c["ta"], c["tb"], m, n, k, 1.5, _ptr(s["A"]), (k if c["ta"] else m) + pad, _ptr(s["B"]),
                             (n if c["tb"] else k) + pad, c["beta"], _ptr(s["C"]), m + pad)
    return s["C"][:, :m]


def _rank_k(s, c, ctx, p):
    n, k, pad, tr = c["n"], c["k"], c["pad"], c["trans"]
    ld = (k if tr else n) + pad
    A, C = _ptr(s["A"]), _ptr(s["C"])
    if c["op"] == "syrk":
        getattr(ctx, p + "syrk")(c["uplo"], tr, n, k, 1.0, A, ld, 0.25, C, n + pad)
    elif c["op"] == "syr2k":
        getattr(ctx, p + "syr2k")(c["uplo"], tr, n, k, 1.0, A, ld, _ptr(s["B"]), ld, 0.25, C, n + pad)
    else:
        getattr(ctx, p + "gemmtr")(c["uplo"], tr, 1 - tr, n, n, k, 1.0, A, ld, _ptr(s["B"]), ld, 0.25, C, n + pad)
    return s["C"][:, :n]


def _symm(s, c, ctx, p):
    m, n, pad = c["m"], c["n"], c["pad"]
    order = m if c["side"] == wg.LEFT else n
    getattr(ctx, p + "symm")(c["side"], c["uplo"], m, n, 1.0, _ptr(s["A"]), order + pad, _ptr(s["B"]), m + pad, 0.5,
                             _ptr(s["C"]), m + pad)
    return s["C"][:, :m]


def _triangular(s, c, ctx, p):
    m, n, pad = c["m"], c["n"], c["pad"]
    order = m if c["side"] == wg.LEFT else n
    X, B = s["X"], s["B"]
    # both routines overwrite their right-hand sides: a program that goes on using B works on a copy
    status = ctx.lib.wgb_memcpy_d2d(ctx.handle, _ptr(X), _ptr(B), B.numel() * B.element_size())
    if status != 0:
        raise RuntimeError("wgb_memcpy_d2d failed with status %d" % status)
    getattr(ctx, p + c["op"])(c["side"], c["uplo"], c["trans"], c["diag"], m, n, 1.0, _ptr(s["A"]), order + pad, _ptr(X), m + pad)
    return X[:, :m]


_RUN = {"reductions": _reductions, "gemv": _gemv, "ger": _ger, "symv": _symv, "trmv": _trmv, "syr2": _syr2, "gemm": _gemm,
        "gemmtr": _rank_k, "syrk": _rank_k, "syr2k": _rank_k, "symm": _symm, "trmm": _triangular, "trsm": _triangular}


# ---- the work that a pass cannot do without -------------------------------------------


def work(c):
    op, e = c["op"], SIZE[c["t"]]
    if op == "reductions":
        n = c["n"]
        return {"bytes": 5 * n * e, "flops": 8 * n}  # dot reads two vectors, the others one each
    if op in ("gemv", "ger"):
        m, n = c["m"], c["n"]
        return {"bytes": ((2 if op == "ger" else 1) * m * n + m + n) * e, "flops": 2 * m * n}
    if op in ("symv", "trmv", "syr2"):
        n = c["n"]
        tri = n * (n + 1) // 2
        return {"bytes": ((2 if op == "syr2" else 1) * tri + 3 * n) * e, "flops": {"symv": 4, "trmv": 2, "syr2": 4}[op] * tri}
    if op == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": (m * k + k * n + (2 if c["beta"] else 1) * m * n) * e, "flops": 2 * m * n * k}
    if op in ("gemmtr", "syrk", "syr2k"):
        n, k = c["n"], c["k"]
        return {"bytes": ((1 if op == "syrk" else 2) * n * k + n * (n + 1)) * e, "flops": (2 if op == "syr2k" else 1) * n * (n + 1) * k}
    m, n = c["m"], c["n"]
    order = m if c["side"] == wg.LEFT else n
    tri = order * (order + 1) // 2
    if op == "symm":
        return {"bytes": (tri + 3 * m * n) * e, "flops": 2 * m * n * order}
    return {"bytes": (tri + 4 * m * n) * e, "flops": m * n * order}  # with the copy of the right-hand sides


# ---- checks --------------------------------------------------------------------------


def tolerance(c):
    """Largest relative error in the 2-norm that a correct implementation at the same precision shows.

    A sum of k products of random signs, in some order, is off by a few units in the last place times
    a slowly growing function of k; the factors are four times what the library was measured at against
    64 (fp32) and 80 (fp64) bits over these ranges, with room for another order of the sums."""
    op, e = c["op"], EPS[c["t"]]
    if op == "reductions":
        # a sequential order within a block's share of up to 65536 elements
        return {"rel": 64 * e, "max": 64 * e}
    if op in ("ger", "syr2"):
        return {"rel": 4 * e, "max": 16 * e}  # three roundings an element
    if op in ("gemv", "symv", "trmv"):
        k = max(c["n"], c.get("m", 0))
    elif op == "gemm":
        k = c["k"]
    elif op in ("gemmtr", "syrk", "syr2k"):
        k = c["k"]
    else:
        k = c["m"] if c["side"] == wg.LEFT else c["n"]
    r = e * max(8.0, math.sqrt(k))
    return {"rel": r, "max": 16 * r}


def _sym(A, n, uplo):
    A = A[:, :n].T  # element (i, j)
    tri = torch.tril(A) if uplo == wg.LOWER else torch.triu(A)
    return tri + tri.T - torch.diag(torch.diagonal(tri))


def _tri(A, n, uplo, diag):
    A = A[:, :n].T
    T = torch.tril(A) if uplo == wg.LOWER else torch.triu(A)
    if diag == wg.UNIT:
        T = T - torch.diag(torch.diagonal(T)) + torch.eye(n, dtype=T.dtype, device=T.device)
    return T


def exact(c, seed):
    """What run() returns for these inputs, in 64 bits, from plain torch."""
    d = {k: v.double() for k, v in _inputs(c, seed).items()}
    op, t = c["op"], c.get("trans", 0)
    if op == "reductions":
        x, y = d["x"][::c["inc"]], d["y"][::c["inc"]]
        dot, asum, nrm2 = (x * y).sum(), x.abs().sum(), x.square().sum().sqrt()
        if c["host"]:
            return {"dot": float(dot), "asum": float(asum), "nrm2": float(nrm2), "index": None}
        return {"sums": torch.stack([dot, asum, nrm2]), "index": None}
    if op == "gemv":
        At = d["A"][:, :c["m"]]
        return 1.5 * ((At if t else At.T) @ d["x"]) + 0.5 * d["y"]
    if op == "ger":
        return d["A"][:, :c["m"]] + 0.75 * torch.outer(d["y"], d["x"])
    if op == "symv":
        return 1.5 * (_sym(d["A"], c["n"], c["uplo"]) @ d["x"]) + 0.5 * d["y"]
    if op == "trmv":
        T = _tri(d["A"], c["n"], c["uplo"], c["diag"])
        return (T.T if t else T) @ d["x"]
    if op == "syr2":
        At = d["A"][:, :c["n"]]
        xy = torch.outer(d["x"], d["y"])
        new = At + 0.75 * (xy + xy.T)
        # At is the transpose: the lower triangle of A is the upper one of At
        keep = torch.ones_like(At, dtype=torch.bool)
        return torch.where(torch.triu(keep) if c["uplo"] == wg.LOWER else torch.tril(keep), new, At)
    if op == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        At = d["A"][:, :k].T if c["ta"] else d["A"][:, :m]  # op(A) transposed, k x m
        Bt = d["B"][:, :n].T if c["tb"] else d["B"][:, :k]  # op(B) transposed, n x k
        return 1.5 * (Bt @ At) + c["beta"] * d["C"][:, :m]
    if op in ("gemmtr", "syrk", "syr2k"):
        n, k = c["n"], c["k"]
        A = d["A"][:, :k] if t else d["A"][:, :n].T  # n x k
        B = A if op == "syrk" else (d["B"][:, :k] if t else d["B"][:, :n].T)
        P = A @ B.T
        if op == "syr2k":
            P = P + P.T
        Ct = d["C"][:, :n]
        keep = torch.ones_like(Ct, dtype=torch.bool)
        return torch.where(torch.triu(keep) if c["uplo"] == wg.LOWER else torch.tril(keep), P.T + 0.25 * Ct, Ct)
    m, n = c["m"], c["n"]
    left = c["side"] == wg.LEFT
    order = m if left else n
    B = d["B"][:, :m].T
    if op == "symm":
        S = _sym(d["A"], order, c["uplo"])
        return (S @ B if left else B @ S).T + 0.5 * d["C"][:, :m]
    T = _tri(d["A"], order, c["uplo"], c["diag"])
    upper = (c["uplo"] == wg.UPPER) != bool(t)
    T = T.T if t else T
    if op == "trmm":
        return (T @ B if left else B @ T).T
    return torch.linalg.solve_triangular(T.contiguous(), B.contiguous(), upper=upper, left=left,
                                         unitriangular=c["diag"] == wg.UNIT).T
