"""Float16 gemm! at the edges of its tiles (64, 128, 256), of its slabs (32)
and of the in-place reading of an operand (16-byte rows, K a multiple of the
slab depth, apart from C).  Small integers: every Float32 partial sum and the
Float16 result are exact, so the product equals the integer one bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def mat(gpu, g, r, c, pad=0, off=0):
    ld = r + pad
    buf = torch.randint(-4, 5, (off + c * ld,), device="cuda", generator=g).half()
    return gpu.DMatrix(buf, r, c, ld, off)


def op(d, t):
    x = d.strided().double().T          # (rows, cols)
    return x.T if t == "T" else x


def check(gpu, m, n, k, ta, tb, beta, pad=(0, 0, 0), off=(0, 0, 0), seed=1):
    g = torch.Generator(device="cuda").manual_seed(seed)
    A = mat(gpu, g, *((k, m) if ta == "T" else (m, k)), pad[0], off[0])
    B = mat(gpu, g, *((n, k) if tb == "T" else (k, n)), pad[1], off[1])
    C = mat(gpu, g, m, n, pad[2], off[2])
    ref = op(A, ta) @ op(B, tb) + beta * op(C, "N")
    outside = C.buf.clone()
    gpu.hgemm_(C, A, B, 1.0, beta, ta, tb)
    assert torch.equal(op(C, "N"), ref)
    C.strided().copy_(torch.zeros_like(C.strided()))
    outside.as_strided(C.strided().shape, C.strided().stride(), C.offset).zero_()
    assert torch.equal(C.buf, outside)     # nothing written between the columns


@pytest.mark.parametrize("ta", "NT")
@pytest.mark.parametrize("tb", "NT")
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (63, 65, 31), (64, 64, 32), (65, 129, 33), (300, 70, 96),
                                   (1800, 1910, 64), (1793, 1792, 33), (3600, 3585, 64), (3584, 3601, 40)])
def test_hgemm_tiles(gpu, m, n, k, ta, tb):
    check(gpu, m, n, k, ta, tb, 0.0)
    check(gpu, m, n, k, ta, tb, 2.0)


@pytest.mark.parametrize("pad,off", [((8, 8, 4), (0, 0, 0)), ((8, 8, 4), (8, 8, 4)), ((1, 8, 0), (0, 0, 0)),
                                     ((0, 0, 0), (1, 0, 0)), ((0, 0, 1), (0, 3, 2)), ((4, 4, 4), (4, 4, 1))])
def test_hgemm_strides_and_offsets(gpu, pad, off):
    for ta, tb in (("T", "N"), ("N", "T")):
        check(gpu, 136, 72, 64, ta, tb, 2.0, pad, off)
        check(gpu, 1800, 1900, 64, ta, tb, 0.0, pad, off)


def test_hgemm_overlapping_operands(gpu):
    g = torch.Generator(device="cuda").manual_seed(3)
    n = 128
    A, B = mat(gpu, g, n, n), mat(gpu, g, n, n)
    for ta, which in (("T", "A"), ("N", "B")):
        a, b = A.copy(), B.copy()
        ref = op(a, ta) @ op(b, "N")
        assert float(ref.abs().max()) <= 2048
        out = gpu.hgemm_(a if which == "A" else b, a, b, 1.0, 0.0, ta, "N")
        assert torch.equal(op(out, "N"), ref)
