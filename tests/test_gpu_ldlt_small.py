"""Batched LDLT for sizes up to 32 (eight lanes per system, the pivot order
found from the diagonal first) against the one-wave-per-system kernel on the
same systems (max_n above 32 selects it): transpositions, sign and info are
equal, and the factors and solutions agree, at every size, on diagonals that
are distinct, tied, zero, partly NaN or infinite, and on singular and
indefinite matrices.

Both kernels take the sums in the same order, so factors may differ by the
contraction of a product and a difference: 8 n eps of the largest entry of |L|
or |D| for the definite kinds; entries of an indefinite or singular factor can
grow by cancellation, where 1e-10 of the largest entry is the bound this
repository's LDLT tests use."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def matrix(rng, kind, n):
    b = rng.standard_normal((n, n))
    if kind == "pos":
        return b @ b.T + n * np.eye(n)
    if kind == "tied":  # a correlation matrix: every diagonal entry is one
        a = b @ b.T + n * np.eye(n)
        d = 1.0 / np.sqrt(np.diag(a))
        a = a * d[:, None] * d[None, :]
        np.fill_diagonal(a, 1.0)
        return a
    if kind == "indef":
        return b + b.T
    if kind == "ints":  # exact arithmetic, repeated magnitudes of both signs
        a = rng.integers(-2, 3, (n, n)).astype(float)
        a = a + a.T
        np.fill_diagonal(a, rng.choice([-8.0, 8.0, 4.0], n) * n)
        return a
    if kind == "zero":
        return np.zeros((n, n))
    if kind == "offdiag":  # zero diagonal, something below it
        a = np.zeros((n, n))
        a[n - 1, 0] = a[0, n - 1] = 1.0
        return a
    if kind == "rank1":
        v = rng.integers(1, 4, n).astype(float)
        return np.outer(v, v)
    if kind == "nan":
        a = b @ b.T + n * np.eye(n)
        a[n // 2, n // 2] = np.nan
        return a
    a = b @ b.T + n * np.eye(n)
    a[n // 3, n // 3] = np.inf
    return a


def run(mats, max_n, rhs):
    from eigen_amd import batched
    n = np.array([m.shape[0] for m in mats])
    offA = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)[:-1]])
    offb = np.concatenate([[0], np.cumsum(n.astype(np.int64))[:-1]])
    d = lambda x, t: torch.tensor(np.ascontiguousarray(x), dtype=t, device="cuda")  # noqa: E731
    A = d(np.concatenate([m.flatten(order="F") for m in mats] + [[3.0]]), torch.float64)
    nn, oa, ob = d(n, torch.int32), d(offA, torch.int64), d(offb, torch.int64)
    T, offT, sign, info = batched.ldlt_batched(oa, nn, A, ob, max_n=max_n)
    x = d(np.concatenate([rhs[:int(n.sum())], [4.0]]), torch.float64)
    batched.ldlt_solve_batched(oa, nn, A, offT, T, ob, x, max_n=max_n)
    return (n, offA, offb, A.cpu().numpy(), T.cpu().numpy(), sign.cpu().numpy(),
            info.cpu().numpy(), x.cpu().numpy())


@pytest.mark.parametrize("kind", ["pos", "tied", "indef", "ints", "zero", "offdiag", "rank1",
                                  "nan", "inf"])
@pytest.mark.parametrize("sizes", [[2, 3, 7, 8], [1, 9, 15, 16, 5], [17, 24, 23, 2, 0, 8, 11],
                                   list(range(1, 33)) + [25, 32, 31]])
def test_against_the_wave_kernel(kind, sizes):
    rng = np.random.default_rng(len(kind) * 100 + len(sizes))
    mats = [matrix(rng, kind, n) if n else np.zeros((0, 0)) for n in sizes]
    rhs = rng.standard_normal(int(sum(sizes)))
    got = run(mats, max(sizes), rhs)
    ref = run(mats, 40, rhs)
    for i in (4, 5, 6):
        assert np.array_equal(got[i], ref[i]), i
    assert got[3][-1] == 3.0 and got[7][-1] == 4.0
    n, offA, offb = got[:3]
    for i, k in enumerate(n):
        if k == 0:
            continue
        f, g = (y[3][offA[i]:offA[i] + k * k].reshape(k, k, order="F") for y in (got, ref))
        assert np.array_equal(np.triu(f, 1), np.triu(g, 1), equal_nan=True)
        f, g = np.tril(f), np.tril(g)
        fin = np.isfinite(g)
        assert np.array_equal(fin, np.isfinite(f))
        top = max(1e-300, np.abs(g[fin]).max(initial=0.0))
        tol = 8 * k * EPS if kind in ("pos", "tied", "ints") else 1e-10
        assert np.all(np.abs(f - g)[fin] <= tol * top), (i, k)
        if kind in ("pos", "tied", "ints"):
            x, y = (z[7][offb[i]:offb[i] + k] for z in (got, ref))
            # condition numbers of these stay below 50 n
            assert np.all(np.abs(x - y) <= 50 * k * 16 * k * EPS * np.abs(y).max())


def test_sizes_outside_and_ragged_count():
    rng = np.random.default_rng(1)
    mats = [matrix(rng, "pos", n) for n in [5, 30, 8, 24] * 5 + [6]]
    rhs = rng.standard_normal(sum(m.shape[0] for m in mats))
    got = run(mats, 24, rhs)
    n, offA, offb = got[:3]
    assert np.array_equal(got[6], np.where(n > 24, -2, 0))
    for i, k in enumerate(n):
        a = mats[i]
        if k > 24:  # left as they were
            assert np.array_equal(got[3][offA[i]:offA[i] + k * k], a.flatten(order="F"))
            assert np.array_equal(got[7][offb[i]:offb[i] + k], rhs[offb[i]:offb[i] + k])
        else:
            x = got[7][offb[i]:offb[i] + k]
            r = rhs[offb[i]:offb[i] + k] - a @ x
            assert np.abs(r).max() <= 1e-14 * (np.abs(a).sum(1).max() * np.abs(x).max() +
                                               np.abs(rhs[offb[i]:offb[i] + k]).max())
