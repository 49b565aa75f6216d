"""Batched LLT rank updates at the edges of the eight-lane kernel (groups of
eight columns, factors up to 32 rows, spans of 32 factors that share a kernel):
every size around them, both storage triangles, updates and downdates mixed in
one wave, a downdate that fails, and sizes the kernel does not take beside
ones it does, each against the oracle's update of the same factor.

Tolerance: an update is n orthogonal (or mildly hyperbolic) rotations applied
to rows of norm below 2 sqrt(2 n): 64 n eps of that norm."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from tests import inputs

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def run(sizes, sig, upper, fail=()):
    from eigen_amd import batched
    sizes = np.asarray(sizes)
    real = np.clip(sizes, 0, 256).astype(np.int64)
    offL = np.concatenate([[0], np.cumsum(real ** 2)[:-1]])
    offv = np.concatenate([[0], np.cumsum(real)[:-1]])
    L = np.full(int((real ** 2).sum()) + 1, 7.0)
    V = np.random.default_rng(3).standard_normal(int(real.sum()) + 1)
    for i, n in enumerate(real):
        f = np.linalg.cholesky(inputs.spd(9000 + i, int(n))) if n else np.zeros((0, 0))
        f = f + np.triu(np.full((n, n), 5.0), 1)  # the other triangle keeps what it holds
        L[offL[i]:offL[i] + n * n] = (f.T if upper else f).flatten(order="F")
        if i in fail:
            V[offv[i]:offv[i] + n] = 0.0
            V[offv[i] + n // 2] = 100.0 * np.sqrt(n)
    Ld = torch.tensor(L, device="cuda")
    info = batched.llt_rank_update_batched(
        torch.tensor(offL, device="cuda"), torch.tensor(sizes, dtype=torch.int32, device="cuda"),
        Ld, torch.tensor(offv, device="cuda"), torch.tensor(V, device="cuda"),
        torch.tensor(sig, dtype=torch.float64, device="cuda"), upper=upper).cpu().numpy()
    out = Ld.cpu().numpy()
    assert out[-1] == 7.0
    for i, n in enumerate(real):
        if sizes[i] < 0 or sizes[i] > 256:
            assert info[i] == -2
            continue
        l0 = L[offL[i]:offL[i] + n * n].reshape(n, n, order="F")
        got = out[offL[i]:offL[i] + n * n].reshape(n, n, order="F")
        if upper:
            l0, got = l0.T, got.T
        ref, rinfo = po.llt_rank_update(np.asfortranarray(l0), V[offv[i]:offv[i] + n], sig[i])
        assert info[i] == rinfo and (rinfo == -1) == (i not in fail)
        tol = 64 * max(n, 1) * EPS * 2 * np.sqrt(2 * max(n, 1))
        assert np.all(np.abs(np.tril(got) - np.tril(ref)) <= tol), (i, n)
        assert np.array_equal(np.triu(got, 1), np.triu(l0, 1))


@pytest.mark.parametrize("upper", [False, True])
@pytest.mark.parametrize("sizes", [
    [1], [8] * 31, [0, 1, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32], [32] * 33,
    list(range(1, 33)) * 3 + [5], [6, 40, 24] * 20, [24] * 40 + [-1, 300] + [9] * 60])
def test_sizes(sizes, upper):
    sig = np.where(np.arange(len(sizes)) % 3 == 1, -0.01, 1.5)
    run(sizes, sig, upper)
    run(sizes, np.full(len(sizes), 0.75), upper)


@pytest.mark.parametrize("n", [2, 9, 24, 32, 50])
def test_failed_downdate_beside_others(n):
    run([n] * 20, np.where(np.arange(20) % 4 == 3, 0.5, -0.01), False, fail=(2, 17))


@pytest.mark.parametrize("copies", [64, 2100, 4200, 8300])
@pytest.mark.parametrize("base", [[0, 1, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 2, 5, 12] * 4,
                                  [3, 1, 2, 33, 5, 2, 9, 40] * 4 + [2, 4, 32, 1] * 8])
def test_counts_that_change_the_launches(base, copies):
    """64 factors, repeated: from 4096 factors on small spans take eight lanes
    per factor, and the other spans one, two, four or eight factors a wave.
    Every copy must come out alike, and the first as the oracle's update."""
    from eigen_amd import batched
    real = np.asarray(base, dtype=np.int64)
    nL, nV = int((real ** 2).sum()), int(real.sum())
    o1 = np.concatenate([[0], np.cumsum(real ** 2)[:-1]])
    o2 = np.concatenate([[0], np.cumsum(real)[:-1]])
    L, V = np.zeros(nL), np.random.default_rng(4).standard_normal(nV)
    for i, n in enumerate(real):
        if n:
            L[o1[i]:o1[i] + n * n] = np.linalg.cholesky(inputs.spd(9100 + i, int(n))).flatten("F")
    sig = np.where(np.arange(64) % 3 == 1, -0.01, 1.5)
    rep = torch.arange(copies, device="cuda")[:, None]
    t = lambda a: torch.tensor(a, device="cuda")
    Ld = t(L).repeat(copies)
    info = batched.llt_rank_update_batched(
        (rep * nL + t(o1)).reshape(-1), t(real.astype(np.int32)).repeat(copies), Ld,
        (rep * nV + t(o2)).reshape(-1), t(V).repeat(copies), t(sig).repeat(copies))
    out = Ld.reshape(copies, nL)
    assert bool((info == -1).all()) and bool((out == out[0]).all())
    got = out[0].cpu().numpy()
    for i, n in enumerate(real):
        l0 = L[o1[i]:o1[i] + n * n].reshape(n, n, order="F")
        ref, _ = po.llt_rank_update(np.asfortranarray(l0), V[o2[i]:o2[i] + n], sig[i])
        tol = 64 * max(n, 1) * EPS * 2 * np.sqrt(2 * max(n, 1))
        g = got[o1[i]:o1[i] + n * n].reshape(n, n, order="F")
        assert np.all(np.abs(np.tril(g) - np.tril(ref)) <= tol), (i, n)
