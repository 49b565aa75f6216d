"""The FP64 U rows of PartialPivLU (the unit lower solve beside each leaf and
each panel): row counts that end inside a 16-row block, column counts that end
inside a wave's sixteen, one to sixteen blocks; an infinity must reach its own
column's rows from its own row on, and nothing else."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from tests import inputs

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def factor(a):
    import eigen_amd as ea
    lu = ea.PartialPivLU(ea.colmajor(torch.from_numpy(np.asfortranarray(a)).cuda()))
    return lu.matrixLU().cpu().numpy(), lu.transpositionsP().cpu().numpy()


@pytest.mark.parametrize("n", [33, 40, 47, 48, 49, 65, 80, 97, 130, 255, 257, 272, 289, 300, 530, 777])
def test_against_the_oracle(n):
    a = inputs.normal(52000 + n, n, n)
    f, t = factor(a)
    ref, t_ref, _, _, margin = po.lu(a, margins=True)
    d = np.nonzero(t != t_ref)[0]
    assert len(d) == 0 or margin[d[0]] < 1e-12
    # backward error of the elimination: n eps times a growth below n
    l, u = np.tril(f, -1) + np.eye(n), np.triu(f)
    p = a.copy()
    for i, j in enumerate(t):
        p[[i, j]] = p[[j, i]]
    assert np.abs(l @ u - p).max() <= n * n * EPS * np.abs(a).max()


@pytest.mark.parametrize("n,row", [(64, 0), (64, 7), (64, 20), (64, 31), (330, 3), (330, 100), (330, 255)])
def test_an_infinity_stays_in_its_column(n, row):
    a = inputs.normal(53000 + n, n, n)
    f, t = factor(a)
    order = np.arange(n)
    for i, j in enumerate(t):
        order[[i, j]] = order[[j, i]]
    b = a.copy()
    b[order[row], n - 1] = np.inf
    g, _ = factor(b)
    # the last column is a candidate for no pivot but its own: the others agree
    assert (g[:, :n - 1] == f[:, :n - 1]).all()
    assert (g[:row, n - 1] == f[:row, n - 1]).all()
    assert g[row, n - 1] == np.inf
    assert not np.isfinite(g[row + 1:, n - 1]).any()
