"""FP64 triangular solves with several right-hand sides (64 x 64 diagonal
blocks inverted, 256 rows per launch, sixteen columns per workgroup) at the
edges of those blocks, for every triangle, transpose, unit diagonal and side.

Tolerance: the triangles have condition numbers below 30 (unit diagonals 1.5
or 1 beside entries of 0.5 / sqrt(n) norm), and both solvers are backward
stable in blocks of 64 with error constants below n: 32 cond n eps max |x|
with cond 30, n capped at the inner block structure's 320."""
import itertools
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -53


def triangle(g, n, pad):
    t = torch.randn(n, n + pad, dtype=torch.float64, generator=g) * (0.5 / math.sqrt(n))
    t = t.t()[:n]
    t.diagonal().add_(1.5)
    return t


@pytest.mark.parametrize("side,uplo,trans,diag",
                         list(itertools.product("LR", "LU", "NT", "NU")))
@pytest.mark.parametrize("n,nrhs", [(1, 2), (33, 3), (63, 16), (64, 17), (65, 2), (255, 5),
                                    (257, 33), (320, 15), (700, 40)])
def test_blocks(n, nrhs, side, uplo, trans, diag):
    import eigen_amd as ea
    g = torch.Generator().manual_seed(n * 131 + nrhs)
    T = triangle(g, n, 1)
    B = torch.randn(nrhs, n, dtype=torch.float64, generator=g).t()
    if side == "R":
        B = torch.randn(n, nrhs, dtype=torch.float64, generator=g).t()
    full = torch.tril(T) if uplo == "L" else torch.triu(T)
    if diag == "U":
        full = full - torch.diag(full.diagonal()) + torch.eye(n, dtype=torch.float64)
    op = full if trans == "N" else full.t()
    ref = torch.linalg.solve(op, B) if side == "L" else torch.linalg.solve(op.t(), B.t()).t()
    X = ea.colmajor(B.cuda()).clone(memory_format=torch.preserve_format)
    Tg = T.cuda()
    Td = torch.empty(n, n + 1, dtype=torch.float64, device="cuda").t()[:n]  # ld = n + 1
    Td.copy_(Tg)
    # the triangle that is not named is not read
    other = torch.triu(torch.ones(n, n), 1) if uplo == "L" else torch.tril(torch.ones(n, n), -1)
    Td[other.bool().cuda()] = float("nan")
    ea.triangular_solve(Td, X, side=side, uplo=uplo, trans=trans, diag=diag)
    tol = 32 * 30 * min(n, 320) * EPS * float(ref.abs().max())
    assert float((X.cpu() - ref).abs().max()) <= tol


def test_columns_do_not_mix():
    """A right-hand side with a NaN or an infinity leaves the others as they are."""
    import eigen_amd as ea
    n = 300
    g = torch.Generator().manual_seed(5)
    T = ea.colmajor(triangle(g, n, 0).cuda())
    B = torch.randn(20, n, dtype=torch.float64, generator=g).t()
    X = ea.colmajor(B.cuda()).clone(memory_format=torch.preserve_format)
    ea.triangular_solve(T, X)
    Bn = B.clone()
    Bn[10, 3], Bn[200, 7] = float("nan"), float("inf")
    Y = ea.colmajor(Bn.cuda()).clone(memory_format=torch.preserve_format)
    ea.triangular_solve(T, Y)
    keep = [c for c in range(20) if c not in (3, 7)]
    assert torch.equal(X[:, keep], Y[:, keep])
    assert bool(torch.isnan(Y[10:, 3]).all()) and not bool(torch.isfinite(Y[200:, 7]).any())
