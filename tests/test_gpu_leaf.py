"""The panel leaf at the sizes where its work division changes: the rows of
one workgroup (256, 512), several workgroups, two rows per thread (257 to 512
and above 8192 rows) and widths 1..64.  Up to 32 columns the leaf's operations
(per column a division, then fma(-l, u, a)) are the oracle's
(src/lapack/factorizations.jl:89-140), so factors, pivots and info are equal
bit for bit; beyond, the oracle halves the columns, and the pivots are
LAPACK's and the reconstruction is within the LU tests' bound."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1), (33, 32), (64, 31), (255, 32), (256, 7), (257, 32), (300, 1), (511, 32), (512, 32), (513, 32),
          (700, 23), (2048, 32), (4100, 32), (8192, 32), (8193, 32), (16500, 32)]


def check(gpu, A):
    F = gpu.lu(gpu.DMatrix.from_numpy(A), check=False)
    Fo, ipo, info = O.dgetrf(A, 128)
    np.testing.assert_array_equal(F.ipiv, ipo)
    assert F.info == info
    np.testing.assert_array_equal(F.factors.numpy(), Fo)


@pytest.mark.parametrize("m,w", SHAPES)
def test_leaf_random_and_ties(gpu, rng, m, w):
    check(gpu, rng.standard_normal((m, w)))
    # few distinct magnitudes: exact ties inside a thread, a wave, a
    # workgroup and between workgroups, and columns that become zero
    check(gpu, rng.integers(-2, 3, (m, w)).astype(np.float64))
    # equal high words, different low words: settled by the low word
    A = 1.0 + rng.integers(0, 1 << 20, (m, w)) * 2.0 ** -52
    check(gpu, A * rng.choice([-1.0, 1.0], (m, w)))


@pytest.mark.parametrize("m,w", [(64, 64), (100, 33), (255, 64), (257, 64), (700, 47), (2048, 64), (8192, 63)])
def test_wide_leaf(gpu, rng, m, w):
    from scipy.linalg.lapack import dgetrf
    A = rng.standard_normal((m, w))
    F = gpu.lu(gpu.DMatrix.from_numpy(A))
    lu, piv, info = dgetrf(A)
    np.testing.assert_array_equal(F.ipiv, piv + 1)
    X = F.factors.numpy()
    L = np.tril(X, -1)
    L[np.arange(w), np.arange(w)] = 1.0
    R = A[F.p - 1] - L @ np.triu(X[:w])
    assert np.linalg.norm(R) <= 30 * w * np.finfo(float).eps * np.linalg.norm(A)
    # a zero column and a NaN row: info of the first, NaN never a pivot below
    # the diagonal
    A[:, w - 2] = 0.0
    A[m - 1, w - 1] = np.nan
    F = gpu.lu(gpu.DMatrix.from_numpy(A), check=False)
    lu, piv, info = dgetrf(A[:, :w - 2])
    assert F.info == w - 1
    np.testing.assert_array_equal(F.ipiv[:w - 2], piv + 1)


@pytest.mark.parametrize("m,w", [(40, 8), (300, 32), (700, 32), (9000, 32)])
def test_leaf_nonfinite_and_zero_pivots(gpu, rng, m, w):
    A = rng.standard_normal((m, w))
    A[:, w // 2] = 0.0                      # a zero pivot in the middle
    A[m // 2, w - 1] = np.inf
    check(gpu, A)
    A = rng.standard_normal((m, w))
    A[m - 1, 1] = np.nan                    # never a pivot below the diagonal
    check(gpu, A)
    A = rng.standard_normal((m, w))
    A[0, 0] = np.nan                        # wins in the diagonal position
    check(gpu, A)


# Interchanges of 64-column panels on the next panel's columns, where the same
# row is reached again and again (a cyclic shift: step s takes the last row every
# time) or rows move about inside the panel and out of it (random permutations,
# with a lower part of the factor that the solve has to apply): exact.
@pytest.mark.parametrize("n", [65, 127, 128, 129, 192, 200, 257, 320, 450])
@pytest.mark.parametrize("kind", ["shift", "back", "random", "scaled"])
def test_interchanges_of_panels_exact(gpu, rng, n, kind):
    if kind == "shift":
        A = np.roll(np.eye(n), 1, axis=1)
    elif kind == "back":
        A = np.roll(np.eye(n), -1, axis=1)
    else:
        # P^T L U with entries that every operation leaves exact
        L = np.tril((rng.integers(-1, 2, (n, n)) * (rng.random((n, n)) < 2.0 / n)).astype(float) * 0.5, -1) + np.eye(n)
        if kind == "random":
            L = np.eye(n)
        A = (L @ np.diag(2.0 ** rng.integers(-2, 3, n)))[rng.permutation(n)]
    for lowp in (False, True):
        M = np.asfortranarray(A.astype(np.float32) if lowp else A)
        F = gpu.lu_lowp(M, "float32", blocksize=64) if lowp else gpu.lu(M, blocksize=64)
        LU = F.factors.numpy().astype(float)
        perm = np.arange(n)
        for i, q in enumerate(F.ipiv_dev.cpu().numpy().astype(int) - 1):
            assert q >= i
            perm[[i, q]] = perm[[q, i]]
        assert np.array_equal((np.tril(LU, -1) + np.eye(n)) @ np.triu(LU), A[perm]), lowp


@pytest.fixture
def own_handle(gpu, monkeypatch):
    """A handle of its own, made under the given environment, in place of the
    device's while the test runs."""
    from oxiblas_mi355x import _lib
    made = []

    def make(**env):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        h = gpu.Handle(0)
        made.append(h)
        monkeypatch.setitem(_lib._handles, 0, h)
        return h
    yield make
    import torch
    torch.cuda.synchronize()
    for h in made:
        h.close()


@pytest.mark.parametrize("n,nb", [(600, 0), (700, 64), (1500, 0), (2600, 128)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_wait_that_gives_up(gpu, rng, own_handle, n, nb, dtype):
    """Leaves whose waits give up at once: the call reports it, pivots that were
    never written are not followed (they name rows far outside), and nothing
    around the matrix changes; one-workgroup factorizations still work."""
    import ctypes as C
    import torch
    h = own_handle(OXIBLAS_LEAF_SPINS="0")
    dt = torch.float64 if dtype == "f64" else torch.float32
    pad, ld = 4096, n + 5
    buf = torch.randn(2 * pad + ld * n, dtype=dt, device="cuda", generator=torch.Generator(device="cuda").manual_seed(n))
    before = buf.clone()
    ipiv = torch.full((n,), 1 << 40, dtype=torch.int64, device="cuda")
    info = C.c_int64(0)
    A = buf.data_ptr() + pad * buf.element_size()
    h.bind_stream(torch.cuda.current_stream().cuda_stream)
    if dtype == "f64":
        rc = h._L.oxi_dgetrf(h.ptr, n, n, A, ld, ipiv.data_ptr(), nb, C.byref(info))
    else:
        rc = h._L.oxi_sgetrf_lowp(h.ptr, 3, n, n, A, ld, ipiv.data_ptr(), nb, C.byref(info))
    assert rc == 5                                       # OXI_ERR_TIMEOUT
    outside = torch.ones(buf.numel(), dtype=torch.bool, device="cuda")
    outside[pad:pad + ld * n].view(n, ld)[:, :n] = False
    assert torch.equal(buf[outside], before[outside])
    check(gpu, rng.standard_normal((300, 32)))


@pytest.mark.parametrize("n", [513, 1000])
def test_exchange_buffer_cleared_between_leaves(gpu, rng, own_handle, n):
    """The exchange buffer cleared after every second leaf, where the tags start
    again: the same factors as without."""
    A = rng.standard_normal((n, n))
    F = gpu.lu(gpu.DMatrix.from_numpy(A))
    F32 = gpu.lu_lowp(A.astype(np.float32), "float32")
    own_handle(OXIBLAS_LEAF_TAGS="2")
    for _ in range(2):
        G = gpu.lu(gpu.DMatrix.from_numpy(A))
        np.testing.assert_array_equal(F.ipiv, G.ipiv)
        np.testing.assert_array_equal(F.factors.numpy(), G.factors.numpy())
        G = gpu.lu_lowp(A.astype(np.float32), "float32")
        np.testing.assert_array_equal(F32.factors.numpy(), G.factors.numpy())


@pytest.mark.parametrize("lowp", [False, True])
@pytest.mark.parametrize("n,width", [(64, 32), (150, 32), (700, 32), (513, 64), (1023, 64), (1100, 128), (2000, 128),
                                     (4500, 128)])
def test_products_summed_before_an_element_rounds(gpu, n, width, lowp):
    """`width` products that together make 1 against an element of 2^53 (2^24):
    subtracted as one sum the element is one less, one by one, or in two halves,
    it stays.  Leaves have 32 columns, panels 64, and 128 from 1024 columns on."""
    big = 2.0 ** 24 if lowp else 2.0 ** 53
    A = np.zeros((n, n), dtype=np.float32 if lowp else np.float64)
    i = np.arange(n)
    A[i, i] = np.where(i < width, 4.0, big)
    A[width:, :width] = 4.0 / width                  # multipliers 1 / width
    A[:width, width:] = 1.0
    F = gpu.lu_lowp(A, "float32") if lowp else gpu.lu(gpu.DMatrix.from_numpy(A))
    assert F.factors.numpy()[width, width] == big - 1.0
