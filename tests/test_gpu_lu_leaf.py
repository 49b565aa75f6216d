"""PartialPivLU's FP64 leaf (rows relabelled instead of moved, pivots found by
the high words of |a| first, one to sixteen workgroups) at the row counts where
its launch changes and on the inputs its search treats apart: equal magnitudes
of both signs, values that differ in the low word only, zero columns,
infinities and NaNs.  Pivots must equal the oracle's; where no candidates tie
within rounding the factors are within n^2 eps of it."""
import numpy as np
import pytest
import torch

from oracle import pyoracle as po
from tests import inputs

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def gpu_lu(a):
    import eigen_amd as ea
    lu = ea.PartialPivLU(ea.colmajor(torch.from_numpy(np.asfortranarray(a)).cuda()))
    return (lu.matrixLU().cpu().numpy(), lu.transpositionsP().cpu().numpy(),
            lu.first_zero_pivot())


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 63, 65, 511, 512, 513, 544, 1023, 1024, 1025,
                               1056, 2050])
def test_launch_edges(n):
    a = inputs.normal(31000 + n, n, n)
    lu, t = gpu_lu(a)[:2]
    ref, t_ref, _, _, margin = po.lu(a, margins=True)
    d = np.nonzero(t != t_ref)[0]
    assert len(d) == 0 or margin[d[0]] < 1e-12
    if len(d) == 0:
        assert np.abs(lu - ref).max() <= n * n * EPS * np.abs(ref).max()


@pytest.mark.parametrize("n", [40, 600, 1100])
def test_exact_ties_take_the_first_row(n):
    """Entries +-1 stay small integers for the first columns: exact ties in
    every column, resolved in row order after the interchanges so far."""
    rng = np.random.default_rng(n)
    a = np.eye(n) * 1.0
    a[:, :6] = rng.choice([-1.0, 1.0], (n, 6))
    lu, t = gpu_lu(a)[:2]
    ref, t_ref = po.lu(a)[:2]
    assert np.array_equal(t[:6], t_ref[:6])
    assert np.array_equal(lu[:, :2], ref[:, :2])


@pytest.mark.parametrize("n", [64, 700, 1300])
def test_low_words_decide(n):
    """Column 0's largest entries share their high word."""
    a = inputs.normal(5, n, n)
    a[:, 0] = 3.0 + np.arange(n) % 37 * 2.0 ** -50
    a[1::2, 0] *= -1.0
    t, t_ref = gpu_lu(a)[1], po.lu(a)[1]
    assert t[0] == t_ref[0]


@pytest.mark.parametrize("n", [50, 530, 1030])
def test_zero_columns_and_non_finite(n):
    a = inputs.normal(6, n, n)
    a[:, 3] = 0.0
    lu, t, fz = gpu_lu(a)
    _, t_ref, fz_ref, _ = po.lu(a)
    assert fz == 3 and t[3] == t_ref[3] == 3
    b = inputs.normal(7, n, n)
    b[n // 2, 0] = np.nan  # a NaN below the diagonal never wins
    assert gpu_lu(b)[1][0] == po.lu(b)[1][0] != n // 2
    b = inputs.normal(8, n, n)
    b[0, 0] = np.nan  # on the diagonal it does, also over an infinity
    b[n - 1, 0] = np.inf
    assert gpu_lu(b)[1][0] == po.lu(b)[1][0] == 0
    b = inputs.normal(9, n, n)
    b[n - 1, 0] = -np.inf
    b[n - 2, 0] = np.inf
    assert gpu_lu(b)[1][0] == po.lu(b)[1][0] == n - 2
