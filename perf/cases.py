"""Timing cases of the level-3 hot path: gemm! in its data types, the batched
product, trsm!, LU with its solve, the solve's backward pass, Cholesky and the
mixed-precision solve, each through the package's public functions.

listed() are the cases that are reported; draw() gives more of the same
ranges; prepare() makes a case's inputs on the GPU from a seed; run() is one
pass; work() counts the bytes and operations a pass cannot do without;
exact() computes the same outputs in 64 bits with torch alone.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxiblas.jl_amd"))

import oxiblas_mi355x as ox  # noqa: E402

_DT = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16}
_GEMM = {"f64": ox.gemm_, "f32": ox.sgemm_, "f16": ox.hgemm_}


def listed():
    return [
        # the reference's medium benchmark size: one product of a small model
        # or a block of a user's own algorithm; launch and latency count
        {"name": "gemm_f64_256", "op": "gemm", "dtype": "f64", "m": 256, "n": 256, "k": 256, "ta": "N", "tb": "N",
         "beta": 0.0},
        # odd sizes, a transposed operand and an accumulated C, as in normal
        # equations and pullbacks
        {"name": "gemm_f64_ragged_tn", "op": "gemm", "dtype": "f64", "m": 1500, "n": 1111, "k": 777, "ta": "T",
         "tb": "N", "beta": 0.5},
        # the large square product
        {"name": "gemm_f64_8192", "op": "gemm", "dtype": "f64", "m": 8192, "n": 8192, "k": 8192, "ta": "N",
         "tb": "N", "beta": 0.0},
        # the Float16 product
        {"name": "gemm_f16_4096", "op": "gemm", "dtype": "f16", "m": 4096, "n": 4096, "k": 4096, "ta": "N",
         "tb": "N", "beta": 0.0},
        # many small products in one call (element matrices, blocks of a
        # block-sparse matrix)
        {"name": "batched_64x1000", "op": "batched", "m": 64, "n": 64, "k": 64, "batch": 1000},
        # a triangular solve with a square right-hand side, as in a user's own
        # blocked factorization or whitening
        {"name": "trsm_2048", "op": "trsm", "m": 2048, "nrhs": 2048, "side": "L", "uplo": "L", "trans": "N"},
        # A \ b from small systems to the headline size; 2000 is no multiple
        # of any block size
        {"name": "lu_solve_256", "op": "lu", "n": 256, "nrhs": 1},
        {"name": "lu_solve_2000", "op": "lu", "n": 2000, "nrhs": 1},
        {"name": "lu_solve_16384", "op": "lu", "n": 16384, "nrhs": 1},
        # forward and backward of X = F \ B on factors that the program keeps
        {"name": "solve_grad_8192", "op": "solve_grad", "n": 8192, "nrhs": 64},
        # a symmetric positive definite system (covariance, normal equations)
        {"name": "cholesky_4096", "op": "cholesky", "n": 4096, "nrhs": 1},
        # Float32 factors refined to FP64 accuracy, the reference's defaults
        {"name": "mixed_4096", "op": "mixed", "n": 4096, "nrhs": 1},
    ]


def _log(rng, lo, hi):
    """A size spread evenly over its logarithm, mostly odd or ragged, a
    quarter of them rounded to a multiple of 32."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.25:
        v -= v % 32
    return max(lo, min(hi, v))


def draw(rng):
    op = rng.choice(("gemm", "gemm", "gemm", "batched", "trsm", "lu", "lu", "solve_grad", "cholesky", "mixed"))
    if op == "gemm":
        return {"op": op, "dtype": rng.choice(("f64", "f64", "f32", "f16")), "m": _log(rng, 32, 8192),
                "n": _log(rng, 32, 8192), "k": _log(rng, 32, 8192), "ta": rng.choice("NT"), "tb": rng.choice("NT"),
                "beta": rng.choice((0.0, 0.5))}
    if op == "batched":
        return {"op": op, "m": _log(rng, 8, 128), "n": _log(rng, 8, 128), "k": _log(rng, 8, 128),
                "batch": _log(rng, 16, 4096)}
    if op == "trsm":
        return {"op": op, "m": _log(rng, 64, 4096), "nrhs": _log(rng, 16, 4096), "side": rng.choice("LR"),
                "uplo": rng.choice("UL"), "trans": rng.choice("NT")}
    if op == "lu":
        return {"op": op, "n": _log(rng, 32, 16384), "nrhs": rng.choice((1, 1, 1, 8, 64))}
    if op == "solve_grad":
        return {"op": op, "n": _log(rng, 128, 8192), "nrhs": _log(rng, 1, 64)}
    if op == "cholesky":
        return {"op": op, "n": _log(rng, 64, 8192), "nrhs": rng.choice((1, 1, 8, 64))}
    return {"op": op, "n": _log(rng, 256, 8192), "nrhs": 1}


# ---------------------------------------------------------------------------
# inputs.  A matrix is held as the torch tensor of its columns: row j of the
# (cols, rows) tensor is column j, the layout DMatrix reads.
# ---------------------------------------------------------------------------
def _randn(g, cols, rows, dtype=torch.float64):
    if dtype == torch.float16:
        return torch.randn(cols, rows, dtype=torch.float32, device="cuda", generator=g).to(dtype)
    return torch.randn(cols, rows, dtype=dtype, device="cuda", generator=g)


def _inputs(case, seed):
    """The case's input tensors, as columns, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    op = case["op"]
    if op == "gemm":
        dt, m, n, k = _DT[case["dtype"]], case["m"], case["n"], case["k"]
        return {"A": _randn(g, m, k, dt) if case["ta"] == "T" else _randn(g, k, m, dt),
                "B": _randn(g, k, n, dt) if case["tb"] == "T" else _randn(g, n, k, dt),
                "C": _randn(g, n, m, dt)}
    if op == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        return {"A": torch.randn(b, k, m, dtype=torch.float64, device="cuda", generator=g),
                "B": torch.randn(b, n, k, dtype=torch.float64, device="cuda", generator=g)}
    if op == "trsm":
        # a triangle whose inverse stays of moderate size: diagonal in [1, 2)
        m = case["m"]
        A = _randn(g, m, m) * (0.5 / math.sqrt(m))
        A.diagonal().copy_(1.0 + torch.rand(m, dtype=torch.float64, device="cuda", generator=g))
        left = case["side"] == "L"
        return {"A": A, "B": _randn(g, case["nrhs"], m) if left else _randn(g, m, case["nrhs"])}
    n, r = case["n"], case["nrhs"]
    if op == "lu":
        return {"A": _randn(g, n, n), "B": _randn(g, r, n)}
    if op == "solve_grad":
        return {"A": _randn(g, n, n), "B": _randn(g, r, n), "Xbar": _randn(g, r, n)}
    if op == "cholesky":
        G = _randn(g, n, n)
        A = (G @ G.T) / n
        A.diagonal().add_(1.0)
        return {"A": A, "B": _randn(g, r, n)}
    A = _randn(g, n, n)                      # mixed: a regular, shifted system
    A.diagonal().add_(2.0 * math.sqrt(n))
    return {"A": A, "B": _randn(g, r, n)}


def _dm(t):
    return ox.DMatrix(t.reshape(-1), t.shape[1], t.shape[0])


def prepare(case, seed):
    x = _inputs(case, seed)
    s = {"case": case}
    if case["op"] == "batched":
        b, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        s["A"] = ox.DBatch(x["A"].reshape(-1), m, k, b)
        s["B"] = ox.DBatch(x["B"].reshape(-1), k, n, b)
        s["C"] = ox.DBatch(torch.empty(b * m * n, dtype=torch.float64, device="cuda"), m, n, b)
        return s
    for name, t in x.items():
        s[name] = _dm(t)
    if case["op"] == "solve_grad":
        s["F"] = ox.lu(s.pop("A"))
    return s


def run(s):
    c = s["case"]
    op = c["op"]
    if op == "gemm":
        return _GEMM[c["dtype"]](s["C"], s["A"], s["B"], 1.0, c["beta"], c["ta"], c["tb"]).buf
    if op == "batched":
        return ox.gemm_strided_batched_(s["C"], s["A"], s["B"]).buf
    if op == "trsm":
        return ox.trsm_(s["B"].copy(), s["A"], 1.0, c["side"], c["uplo"], c["trans"]).buf
    if op == "lu":
        F = ox.lu(s["A"])
        return {"factors": F.factors.buf, "ipiv": F.ipiv_dev, "x": F.solve(s["B"]).buf}
    if op == "solve_grad":
        X = s["F"].solve(s["B"])
        Abar, Bbar = ox.ldiv_pullback(s["F"], X, s["Xbar"])
        return {"x": X.buf, "Abar": Abar.buf, "Bbar": Bbar.buf}
    if op == "cholesky":
        F = ox.cholesky(s["A"])
        return {"factors": F.factors.buf, "x": F.solve(s["B"]).buf}
    return ox.mixed_solve(s["A"], s["B"]).x.buf


def work(case):
    op = case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        size = {"f64": 8, "f32": 4, "f16": 2}[case["dtype"]]
        return {"bytes": size * (m * k + k * n + m * n * (2 if case["beta"] else 1)), "flops": 2 * m * n * k}
    if op == "batched":
        m, n, k, b = case["m"], case["n"], case["k"], case["batch"]
        return {"bytes": 8 * b * (m * k + k * n + m * n), "flops": 2 * m * n * k * b}
    if op == "trsm":
        m, r = case["m"], case["nrhs"]
        return {"bytes": 8 * (m * m // 2 + 2 * m * r), "flops": m * m * r}
    n, r = case["n"], case["nrhs"]
    if op == "lu":
        return {"bytes": 8 * (2 * n * n + 2 * n * r + n), "flops": 2 * n ** 3 // 3 + 2 * n * n * r}
    if op == "solve_grad":
        return {"bytes": 8 * (2 * n * n + 4 * n * r), "flops": 6 * n * n * r}
    if op == "cholesky":
        return {"bytes": 8 * (n * n // 2 + n * n + 2 * n * r), "flops": n ** 3 // 3 + 2 * n * n * r}
    return {"bytes": 8 * (n * n + 2 * n), "flops": 2 * n ** 3 // 3 + 2 * n * n}


def exact(case, seed):
    x = {k: v.double() for k, v in _inputs(case, seed).items()}
    op = case["op"]
    if op == "gemm":
        # columns of C = rows of C^T = op(B)^T op(A)^T; an operand's tensor is its transpose
        At = x["A"].T if case["ta"] == "T" else x["A"]
        Bt = x["B"].T if case["tb"] == "T" else x["B"]
        Ct = Bt.contiguous() @ At.contiguous()
        return (Ct + case["beta"] * x["C"] if case["beta"] else Ct).reshape(-1)
    if op == "batched":
        return torch.bmm(x["B"], x["A"]).reshape(-1)
    if op == "trsm":
        A = x["A"].T
        T = torch.triu(A) if case["uplo"] == "U" else torch.tril(A)
        upper = case["uplo"] == "U"
        if case["trans"] == "T":
            T, upper = T.T, not upper
        X = torch.linalg.solve_triangular(T.contiguous(), x["B"].T.contiguous(), upper=upper,
                                          left=case["side"] == "L")
        return X.T.contiguous().reshape(-1)
    A, B = x["A"].T, x["B"].T
    if op == "lu":
        # the factors by LAPACK on the host, whose pivots are the reference's
        # (up to the size that takes seconds); the solution on the GPU
        factors = torch.linalg.lu_factor(A.cpu())[0].T.contiguous().reshape(-1) if case["n"] <= 8192 else None
        X = torch.linalg.solve(A, B.contiguous())
        return {"factors": factors, "ipiv": None, "x": X.T.contiguous().reshape(-1)}
    if op == "solve_grad":
        LU, piv = torch.linalg.lu_factor(A)
        X = torch.linalg.lu_solve(LU, piv, B.contiguous())
        Bbar = torch.linalg.lu_solve(LU, piv, x["Xbar"].T.contiguous(), adjoint=True)
        Abar_cols = -(X @ Bbar.T)            # columns of Abar = -Bbar X^T
        return {"x": X.T.contiguous().reshape(-1), "Abar": Abar_cols.contiguous().reshape(-1),
                "Bbar": Bbar.T.contiguous().reshape(-1)}
    if op == "cholesky":
        L = torch.linalg.cholesky(A)
        X = torch.cholesky_solve(B.contiguous(), L)
        return {"factors": L.T.contiguous().reshape(-1), "x": X.T.contiguous().reshape(-1)}
    return torch.linalg.solve(A, B.contiguous()).T.contiguous().reshape(-1)
