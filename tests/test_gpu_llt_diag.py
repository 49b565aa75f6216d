"""The Cholesky diagonal block (32-column sub-blocks on lanes in rows of
sixteen) at the edges of its rows, sub-blocks and blocks: the factor against
the oracle, the column a failure is reported at, and a NaN, which passes the
reference's `x <= 0` and must stay in its own row and column."""
import numpy as np
import pytest
import torch

import eigen_amd as ea
from oracle import pyoracle as po
from tests import inputs

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def factor(a):
    f = ea.LLT(ea.colmajor(torch.from_numpy(np.asfortranarray(a)).cuda()))
    return np.tril(f.matrixLLT().cpu().numpy()), f.info()


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 95, 96, 97,
                               127, 128, 129, 160, 200, 257])
def test_edges(n):
    a = inputs.spd(54000 + n, n)
    l, info = factor(a)
    assert info == ea.Success
    # the elimination's backward error: (n + 1) eps |L| |L^T| entrywise, with
    # the row sums of squares at most max |a|
    assert np.abs(l @ l.T - a).max() <= 4 * (n + 1) * EPS * np.abs(a).max()
    ref, _ = po.llt(a)
    cond = np.linalg.cond(a)
    assert np.abs(l - np.tril(ref)).max() <= 8 * n * EPS * cond * np.abs(ref).max()


@pytest.mark.parametrize("bad", [0, 1, 15, 16, 17, 31, 32, 47, 48, 63, 64, 100, 127, 128, 140])
def test_failure_is_reported(bad):
    n = 150
    a = inputs.spd(55000 + bad, n)
    a[bad, bad] = -a[bad, bad]
    assert factor(a)[1] == ea.NumericalIssue
    assert po.llt(a)[1] == bad


@pytest.mark.parametrize("row,col", [(40, 3), (40, 20), (100, 17), (127, 126)])
def test_a_nan_stays_in_its_row_and_column(row, col):
    n = 128
    a = inputs.spd(56000 + row, n)
    l0 = factor(a)[0]
    b = a.copy()
    b[row, col] = b[col, row] = np.nan
    l, info = factor(b)
    assert info == ea.Success
    # before column `col` nothing differs; rows above `row` never do
    assert (l[:, :col] == l0[:, :col]).all() and (l[:row] == l0[:row]).all()
    assert np.isnan(l[row, col:row + 1]).all() and np.isnan(l[row + 1:, row]).all()
    # other rows are untouched up to column row - 1
    assert (l[row + 1:, :row] == l0[row + 1:, :row]).all()
