"""trsm! on the GPU (oxi_dtrsm through the C ABI) against the oracle's
restatement of src/blas/level3.jl:518-544, every side / uplo / trans / diag,
widths that hit each leaf variant (8, 16, 32, 64 and others) and the
recursive split above 64."""
import itertools

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def tri(rng, n, uplo, unit):
    T = rng.standard_normal((n, n)) / max(n, 1) + 2.0 * np.eye(n)
    T = np.triu(T) if uplo == "U" else np.tril(T)
    return np.asfortranarray(T)   # a unit solve ignores the diagonal


@pytest.mark.parametrize("side,uplo,trans,diag", list(itertools.product("LR", "UL", "NT", "NU")))
def test_trsm_all_variants_vs_oracle(gpu, rng, side, uplo, trans, diag):
    for n, other in ((1, 5), (5, 3), (8, 70), (16, 33), (32, 129), (33, 7), (64, 300), (100, 65), (129, 40),
                     (256, 1000)):
        T = tri(rng, n, uplo, diag == "U")
        m, k = (n, other) if side == "L" else (other, n)
        B = np.asfortranarray(rng.standard_normal((m, k)))
        alpha = 0.75
        X = gpu.trsm_(B.copy(order="F"), T, alpha, side, uplo, trans, diag == "U")
        Xo = B.copy(order="F")
        assert O.dtrsm(Xo, T, alpha, side, uplo, trans, diag == "U") == 0
        scale = np.abs(Xo).max() + 1e-300
        assert np.abs(X - Xo).max() <= 1e-12 * scale * max(n, 1), (side, uplo, trans, diag, n, other)


def test_trsm_right_tall(gpu, rng):
    # the shape of U12 = A12 * (L11^T)^-1 in getrf's working layout: many rows, 256 columns
    n, rows = 256, 5000
    T = tri(rng, n, "U", True)
    B = np.asfortranarray(rng.standard_normal((rows, n)))
    X = gpu.trsm_(B.copy(order="F"), T, 1.0, "R", "U", "N", True)
    Xo = B.copy(order="F")
    assert O.dtrsm(Xo, T, 1.0, "R", "U", "N", True) == 0
    assert np.abs(X - Xo).max() <= 1e-11 * np.abs(Xo).max()


@pytest.mark.parametrize("uplo,trans,diag", list(itertools.product("UL", "NT", "NU")))
def test_trsm_right_tall_all_variants(gpu, rng, uplo, trans, diag):
    """Right-side solves with 1500 rows: when op(T) is upper and n a multiple
    of 64 they invert op(T)'s 64 x 64 diagonal blocks and replace each
    64-column sweep by an in-place block product; n = 100 and the lower op(T)
    keep the column sweeps."""
    for n in (64, 192, 320, 100):
        T = tri(rng, n, uplo, diag == "U")
        B = np.asfortranarray(rng.standard_normal((1500, n)))
        X = gpu.trsm_(B.copy(order="F"), T, -0.5, "R", uplo, trans, diag == "U")
        Xo = B.copy(order="F")
        assert O.dtrsm(Xo, T, -0.5, "R", uplo, trans, diag == "U") == 0
        scale = np.abs(Xo).max() + 1e-300
        assert np.abs(X - Xo).max() <= 1e-12 * scale * n, (uplo, trans, diag, n)


def test_trsm_singular_reported_before_write(gpu, rng):
    T = tri(rng, 20, "U", False)
    T[7, 7] = 0.0
    B = np.asfortranarray(rng.standard_normal((20, 3)))
    B0 = B.copy()
    with pytest.raises(gpu.SingularException) as e:
        gpu.trsm_(B, T, 1.0, "L", "U", "N", False)
    assert e.value.info == 8
    assert np.array_equal(B, B0)


# Solves through the inverted diagonal blocks (128 rows for one right-hand
# side, 64 for several) at the edges of the blocks and of their 16-wide tiles.
# Backward error of LU or Cholesky plus two triangular solves: at most a small
# multiple of n eps (|A| |x| + |b|), 4 for each of the factorization and the
# solves, of well-conditioned blocks.
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 144, 255, 257, 385])
@pytest.mark.parametrize("nrhs", [1, 3, 40])
def test_block_inverse_solves(gpu, rng, n, nrhs):
    A = rng.standard_normal((n, n)) + 2.0 * np.sqrt(n) * np.eye(n)
    B = np.asfortranarray(rng.standard_normal((n, nrhs)))
    S = A @ A.T + n * np.eye(n)

    def residual(M, X, eps):
        r = np.linalg.norm(M @ X - B)
        assert r <= 8 * max(n, 8) * eps * (np.linalg.norm(M) * np.linalg.norm(X) + np.linalg.norm(B)), r
    F = gpu.lu(np.asfortranarray(A))
    for t in "NT":
        residual(A if t == "N" else A.T, F.solve(B, t), EPS)
        residual(A if t == "N" else A.T, F.solve(B, t), EPS)      # the second solve runs on a kept plan
    residual(S, gpu.cholesky(np.asfortranarray(S)).solve(B), EPS)
    F32 = gpu.lu_lowp(np.asfortranarray(A.astype(np.float32)), "float32")
    for t in "NT":
        X = F32.solve(np.asfortranarray(B.astype(np.float32)), t)
        X = X.numpy() if hasattr(X, "numpy") else X
        residual((A if t == "N" else A.T).astype(np.float32).astype(float), X.astype(float), np.finfo(np.float32).eps)


# Blocks of 256 rows, full ones and a last one of fewer, on either side, against
# op(A) X = B (X op(A) = B): a backward error of at most 8 n eps, blocks well
# conditioned; 8400 rows are more than the buffer of block inverses holds.
@pytest.mark.parametrize("side,uplo,trans,diag", list(itertools.product("LR", "UL", "NT", "NU")))
@pytest.mark.parametrize("n,other", [(129, 16), (191, 40), (512, 16), (513, 33), (600, 17), (640, 300), (1023, 129)])
def test_trsm_blocked_edges(gpu, side, uplo, trans, diag, n, other):
    _blocked(gpu, side, uplo, trans, diag, n, other)


@pytest.mark.parametrize("side", "LR")
@pytest.mark.parametrize("uplo", "LU")
def test_trsm_blocked_large(gpu, side, uplo):
    _blocked(gpu, side, uplo, "N", "N", 8400, 24)


def _blocked(gpu, side, uplo, trans, diag, n, other):
    import torch
    g = torch.Generator(device="cuda").manual_seed(n + other)
    ld = n + 3
    A = torch.randn(n, ld, dtype=torch.float64, device="cuda", generator=g) / n      # A[c][r]; the other triangle is noise
    A[:, :n].diagonal().copy_(1.0 + torch.rand(n, dtype=torch.float64, device="cuda", generator=g))
    m, k = (n, other) if side == "L" else (other, n)
    B = torch.randn(k, m + 1, dtype=torch.float64, device="cuda", generator=g)
    B0 = B.clone()
    gpu.trsm_(gpu.DMatrix(B.view(-1), m, k, m + 1), gpu.DMatrix(A.view(-1), n, n, ld), side=side, uplo=uplo, trans=trans,
              unit=diag == "U")
    T = A[:, :n].T
    T = torch.tril(T) if uplo == "L" else torch.triu(T)
    if diag == "U":
        T = T - torch.diag(T.diagonal()) + torch.eye(n, dtype=torch.float64, device="cuda")
    T = (T.T if trans == "T" else T).contiguous()
    X, R = B[:, :m].T.contiguous(), B0[:, :m].T
    r = (T @ X if side == "L" else X @ T) - R
    assert r.norm() <= 8 * n * EPS * (T.norm() * X.norm() + R.norm())
    assert torch.equal(B[:, m], B0[:, m])


# What a substitution leaves finite stays finite.  An infinity (NaN) in B reaches
# the rows solved after it and no others, in its own right-hand side alone; a
# triangle whose block inverses overflow (2^17 below a unit diagonal), or where a
# reciprocal of the diagonal does, still gives what the substitution gives.
VARIANTS = list(itertools.product("LR", "UL", "NT", "NU"))


def oracle_trsm(B, T, side, uplo, trans, diag):
    Xo = B.copy(order="F")
    with np.errstate(all="ignore"):
        assert O.dtrsm(Xo, T, 1.0, side, uplo, trans, diag == "U") == 0
    return Xo


@pytest.mark.parametrize("side,uplo,trans,diag", VARIANTS)
@pytest.mark.parametrize("n,other", [(129, 16), (130, 33), (513, 20)])
def test_trsm_nonfinite_right_hand_sides(gpu, rng, side, uplo, trans, diag, n, other):
    T = tri(rng, n, uplo, diag == "U")
    m, k = (n, other) if side == "L" else (other, n)
    B = np.asfortranarray(rng.standard_normal((m, k)))
    Bs = B if side == "L" else B.T                  # right-hand sides as columns, in place
    Bs[100, 3] = np.inf
    Bs[20, 7] = np.nan
    Bs[n - 1, 15] = -np.inf
    Xo = oracle_trsm(B, T, side, uplo, trans, diag)
    X = gpu.trsm_(B.copy(order="F"), T, 1.0, side, uplo, trans, diag == "U")
    fin = np.isfinite(Xo)
    assert 0 < (~fin).sum() < 3 * n
    np.testing.assert_array_equal(np.isfinite(X), fin)
    assert np.abs(X[fin] - Xo[fin]).max() <= 1e-12 * np.abs(Xo[fin]).max() * n


@pytest.mark.parametrize("side,uplo,trans,diag", VARIANTS)
@pytest.mark.parametrize("n,other", [(129, 16), (256, 17), (513, 40)])
def test_trsm_inverses_out_of_range(gpu, rng, side, uplo, trans, diag, n, other):
    m, k = (n, other) if side == "L" else (other, n)
    off = 1 if uplo == "U" else -1

    def exact(T, X):
        op = T.T if trans == "T" else T
        B = np.asfortranarray(op @ X if side == "L" else X @ op)      # sums of two numbers: exact
        np.testing.assert_array_equal(gpu.trsm_(B, np.asfortranarray(T), 1.0, side, uplo, trans, diag == "U"), X)
    exact(np.eye(n) + 2.0 ** 17 * np.eye(n, k=off), np.ones((m, k)))
    if diag == "N":                                  # 2^-1070: its reciprocal is infinite
        T = np.eye(n) + np.eye(n, k=off)
        T[77, 77] = 2.0 ** -1070
        X = rng.integers(-4, 5, (m, k)).astype(float)
        if side == "L":
            X[76:79:2] = 0.0
        else:
            X[:, 76:79:2] = 0.0
        T[77, 77 + off] = T[77 - off, 77] = 0.0
        exact(T, X)


@pytest.mark.parametrize("side,uplo,trans,diag", VARIANTS)
def test_trsm_graded_triangles(gpu, rng, side, uplo, trans, diag):
    """Columns (rows) falling by 10^-27 and more over a block: the componentwise
    backward error of a substitution, at most (n + 2) unit roundoffs."""
    n, other = 200, 24
    for grade in (-0.5, 0.5):
        for by_rows in (False, True):
            T = rng.standard_normal((n, n)) / 8 + np.diag(1.0 + rng.random(n))
            g = 10.0 ** (grade * np.arange(n))
            T = np.asfortranarray(g[:, None] * T if by_rows else T * g)
            T = np.triu(T) if uplo == "U" else np.tril(T)
            if diag == "U":
                T = np.asfortranarray(T / (T.diagonal()[:, None] if by_rows else T.diagonal()[None, :]))
            m, k = (n, other) if side == "L" else (other, n)
            B = np.asfortranarray(rng.standard_normal((m, k)))
            X = gpu.trsm_(B.copy(order="F"), np.asfortranarray(T), 1.0, side, uplo, trans, diag == "U")
            op = (T.T if trans == "T" else T).astype(np.longdouble)
            if side == "R":
                op, X, B = op.T, X.T, B.T
            fin = np.isfinite(X).all(axis=0) & (np.abs(X) < 1e280).all(axis=0)
            X, B = X[:, fin].astype(np.longdouble), B[:, fin]
            assert fin.any()
            R = np.abs(op @ X - B)
            assert (R <= (n + 2) * (EPS / 2) * (np.abs(op) @ np.abs(X) + np.abs(B))).all()


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("n,i,k", [(100, 50, 53), (200, 100, 103), (200, 150, 163), (385, 300, 301)])
@pytest.mark.parametrize("nrhs", [1, 8])
@pytest.mark.parametrize("lowp", [False, True])
def test_solve_with_nonfinite_factor(gpu, rng, value, n, i, k, nrhs, lowp):
    """U(i, k) not finite, inside a diagonal block that the solves invert: rows
    i + 1 on of x do not depend on it and are what substitution gives, rows up
    to i are not finite.  (L is the identity.)"""
    A = np.triu(rng.standard_normal((n, n)) / n) + np.diag(1.0 + rng.random(n))
    A = np.asfortranarray(A.astype(np.float32) if lowp else A)
    F = gpu.lu_lowp(A, "float32") if lowp else gpu.lu(A)
    F.factors.buf[F.factors.offset + i + k * F.factors.ld] = value
    B = np.asfortranarray(rng.standard_normal((n, nrhs)).astype(A.dtype))
    X = F.solve(B)
    X = X.numpy() if hasattr(X, "numpy") else X
    assert not np.isfinite(X[:i + 1]).any()
    assert np.isfinite(X[i + 1:]).all()
    R = A[i + 1:, i + 1:].astype(float) @ X[i + 1:].astype(float) - B[i + 1:]
    eps = np.finfo(A.dtype).eps
    assert np.linalg.norm(R) <= 8 * n * eps * (np.linalg.norm(A) * np.linalg.norm(X[i + 1:]) + np.linalg.norm(B))


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("side,uplo,trans", list(itertools.product("LR", "UL", "NT")))
@pytest.mark.parametrize("n,other", [(200, 24), (512, 24), (512, 700)])
def test_trsm_nonfinite_triangle(gpu, rng, value, side, uplo, trans, n, other):
    """An element of the triangle that is not finite, inside a 16 x 16 tile of a
    diagonal block: what is solved before its row is finite and right."""
    T = tri(rng, n, uplo, False)
    lo, hi = 101, 107
    T0 = T.copy()
    T[(lo, hi) if uplo == "U" else (hi, lo)] = value
    m, k = (n, other) if side == "L" else (other, n)
    B = np.asfortranarray(rng.standard_normal((m, k)))
    X = gpu.trsm_(B.copy(order="F"), T, 1.0, side, uplo, trans)
    Xo = oracle_trsm(B, T0, side, uplo, trans, "N")
    if side == "R":
        X, Xo = X.T, Xo.T
    up = (uplo == "U") ^ (trans == "T") ^ (side == "R")       # solved from the last row (column) up
    first, rest = (slice(lo + 1, None), slice(None, lo + 1)) if up else (slice(None, hi), slice(hi, None))
    assert not np.isfinite(X[rest]).any() and np.isfinite(X[first]).all()
    assert np.abs(X[first] - Xo[first]).max() <= 1e-12 * np.abs(Xo[first]).max() * n


@pytest.mark.parametrize("side", "LR")
def test_solves_on_two_streams(gpu, side):
    """Calls of one handle on two streams, the second enqueued while the first
    runs: each gives what it gives alone.  Then a factorization on the second."""
    import torch

    def make(n, other, seed):
        g = torch.Generator(device="cuda").manual_seed(seed)
        A = torch.randn(n, n, dtype=torch.float64, device="cuda", generator=g) / n
        B = torch.randn(other * n, dtype=torch.float64, device="cuda", generator=g)
        return gpu.DMatrix(A.view(-1), n, n), gpu.DMatrix(B, *((n, other) if side == "L" else (other, n)))

    def solve(A, B, uplo):
        return gpu.trsm_(B, A, 1.0, side, uplo, "N", True).buf       # a unit diagonal: no synchronisation
    A1, B1 = make(4001, 3000, 1)
    A2, B2 = make(1500, 300, 2)
    S = A2.copy()
    S.strided().copy_(S.strided() @ S.strided().T + torch.eye(1500, dtype=torch.float64, device="cuda"))
    want1, want2 = solve(A1, B1.copy(), "L"), solve(A2, B2.copy(), "U")
    wantC = gpu.cholesky(S).factors.buf
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for chol in (False, True):
        X1, X2 = B1.copy(), B2.copy()
        torch.cuda.synchronize()
        with torch.cuda.stream(s1):
            got1 = solve(A1, X1, "L")
        with torch.cuda.stream(s2):
            got2 = gpu.cholesky(S).factors.buf if chol else solve(A2, X2, "U")
        torch.cuda.synchronize()
        assert torch.equal(got1, want1) and torch.equal(got2, wantC if chol else want2)


@pytest.mark.parametrize("n,other", [(200, 100), (600, 40)])
def test_captured_solve(gpu, n, other):
    """A solve with a unit diagonal neither synchronises nor allocates: captured
    into a graph, each replay gives what the call gives, with calls between."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(n)
    A = gpu.DMatrix(torch.randn(n * n, dtype=torch.float64, device="cuda", generator=g) / n, n, n)
    B = torch.randn(n * other, dtype=torch.float64, device="cuda", generator=g)
    X = gpu.DMatrix(B.clone(), n, other)

    def solve(M):
        return gpu.trsm_(M, A, 1.0, "L", "L", "N", True).buf
    want = solve(gpu.DMatrix(B.clone(), n, other)).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        solve(X)
    for _ in range(3):
        X.buf.copy_(B)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(X.buf, want)
        assert torch.equal(solve(gpu.DMatrix(B.clone(), n, other)), want)
        torch.cuda.synchronize()
