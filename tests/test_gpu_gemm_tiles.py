"""FP64 GEMM / SYRK at the edges of its tiles (16, 32, 64 and 128 wide, K slabs
of 16, 32 and 64): remainders in every dimension, one-row operands, leading
dimensions beyond the rows and operands that start 8 bytes off a 16-byte
boundary, against torch's FP64 product on the CPU.

Tolerance, per element: a K-term dot product in any order is within
(K + 2) eps of the exact one relative to sum |a_i b_i| (+ |beta c|), and so is
the reference's."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


def operand(g, rows, cols, off):
    """A column-major rows x cols view, `off` rows into a taller buffer."""
    t = torch.randn(cols, rows + off + 1, dtype=torch.float64, generator=g)
    return t.cuda().t()[off:off + rows]


def check(m, n, k, ta, tb, alpha, beta, off=1):
    import eigen_amd as ea
    g = torch.Generator().manual_seed(m * 1000003 + n * 1009 + k)
    A = operand(g, *((m, k) if ta == "N" else (k, m)), off)
    B = operand(g, *((k, n) if tb == "N" else (n, k)), 0)
    C = operand(g, m, n, off)
    a, b, c = A.cpu(), B.cpu(), C.cpu()
    a, b = (a if ta == "N" else a.t()), (b if tb == "N" else b.t())
    if beta == 0.0:
        C.fill_(float("nan"))  # BLAS: beta = 0 does not read C
    out = ea.gemm(A, B, C, alpha=alpha, beta=beta, transa=ta, transb=tb).cpu()
    ref = alpha * (a @ b) + (beta * c if beta else 0.0)
    bound = 2 * (k + 4) * EPS * (abs(alpha) * (a.abs() @ b.abs()) + abs(beta) * c.abs())
    assert bool(((out - ref).abs() <= bound).all())


@pytest.mark.parametrize("ta,tb", list(itertools.product("NT", "NT")))
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (1, 300, 200), (300, 1, 200), (17, 33, 5), (16, 16, 4001), (50, 31, 1000),  # 16
    (17, 4000, 33), (400, 401, 63), (33, 4100, 129),                                       # 32
    (1025, 1000, 31), (1023, 900, 97), (2000, 513, 65),                                    # 64
    (2049, 2047, 17), (1921, 2111, 127), (4000, 2001, 1)])                                 # 128
def test_tile_edges(m, n, k, ta, tb):
    check(m, n, k, ta, tb, 1.0, 0.0)
    check(m, n, k, ta, tb, -0.5, 2.0, off=0)


@pytest.mark.parametrize("ta,tb", list(itertools.product("NT", "NT")))
@pytest.mark.parametrize("k", [112, 128, 144, 256])
def test_update_reads_c_beside_k(k, ta, tb):
    """alpha = -1, beta = 1 on 128-wide tiles: whole and partial ones, and K
    one slab under, at and past the eight that carry C."""
    check(2305, 2048, k, ta, tb, -1.0, 1.0)
    check(2176, 2049, k, ta, tb, 1.0, 1.0, off=0)


@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("n,k", [(1, 3), (63, 65), (65, 17), (700, 33), (2500, 128), (4225, 130)])
def test_rank_update_tiles(n, k, uplo):
    import eigen_amd as ea
    g = torch.Generator().manual_seed(n + k)
    A = operand(g, n, k, 1)
    C = ea.colmajor(torch.randn(n, n, dtype=torch.float64, generator=g).cuda()).clone()
    C = ea.colmajor(C)
    c, a = C.cpu(), A.cpu()
    ea.rank_update(C, A, alpha=-1.0, uplo=uplo, beta=1.0)
    keep = torch.tril if uplo == "L" else torch.triu
    ref = keep(c - a @ a.t()) + (c - keep(c))
    bound = 2 * (k + 4) * EPS * (a.abs() @ a.abs().t() + c.abs())
    assert bool(((C.cpu() - ref).abs() <= bound).all())
