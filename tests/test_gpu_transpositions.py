"""The right-hand side's row interchanges: with identity factors dgetrs returns
the permuted right-hand side, exactly, in both directions; sequences whose
steps touch each other's rows (as the last rows of every factorization do,
and all of them for tiny orders), that go back to earlier rows, and that touch
one row over and over; columns in LDS and beyond."""
import ctypes as C

import numpy as np
import pytest
import torch

from eigen_amd import dense
from eigen_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def sequences(n, rng):
    k = np.arange(n)
    yield "pivots", k + (rng.random(n) * (n - k)).astype(np.int64)
    yield "anywhere", rng.integers(0, n, n)
    yield "one row", np.full(n, n - 1)
    yield "next row", np.minimum(k + 1, n - 1)
    yield "same mark", np.minimum(k + 1024, n - 1)
    yield "none", k


@pytest.mark.parametrize("n", [1, 2, 3, 63, 64, 65, 127, 128, 129, 500, 1025, 3000, 18432, 18433])
def test_both_directions(n):
    print(f"n={n}", flush=True)
    rng = np.random.default_rng(n)
    eye = torch.eye(n, dtype=torch.float64, device="cuda")
    for nrhs in (1, 3):
        for name, t in sequences(n, rng):
            order = np.arange(n)
            for i, j in enumerate(t):
                order[[i, j]] = order[[j, i]]
            b = rng.standard_normal((n, nrhs))
            td = torch.tensor(t.astype(np.int32), device="cuda")
            for trans in (b"N", b"T"):
                x = dense.colmajor(torch.from_numpy(np.asfortranarray(b)))
                check("eamd_dgetrs", lib().eamd_dgetrs(
                    dense.handle(), trans, n, nrhs, C.c_void_p(eye.data_ptr()), n,
                    C.c_void_p(td.data_ptr()), C.c_void_p(x.data_ptr()), n))
                want = np.empty_like(b)
                if trans == b"N":
                    want[:] = b[order]
                else:
                    want[order] = b
                assert np.array_equal(x.cpu().numpy(), want), (name, trans, nrhs)
