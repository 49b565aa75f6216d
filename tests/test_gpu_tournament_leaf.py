"""The FP32 leaf's tournament at the row counts where its rounds change: two
groups with a last one of a single row, nine groups (the wider final round),
groups of 512 and of 1024 rows, and a merge round before the final one; leading
dimensions with and without 16-byte rows, last leaves narrower than 32.

The matrix is a row-permuted Householder reflection, condition 1 and with zeros
nowhere on its path to need luck: with an FP32 factor of relative error e0 the
solution after one refinement step is off by about e0^2 (the FP64 residual adds
1e-16), and e0 <= 10 n u32 leaves a factor of ten for the growth of the
elimination.  A factor with a row out of place has e0 of order one."""
import numpy as np
import pytest
import torch

from eigen_amd import mixed

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("n", [257, 260, 289, 2048, 2049, 2084, 4097, 4100, 8193, 8228, 16420])
def test_one_refinement_step(n):
    print(f"n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    v = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    perm = torch.randperm(n, device="cuda", generator=g)
    a = torch.eye(n, dtype=torch.float64, device="cuda")[perm]
    a -= (2.0 / (v @ v)) * torch.outer(v[perm], v)
    b = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    a = a.t().contiguous().t()
    x, rep = mixed.gesv_ir(a, b, precision="fp32", check_converged=False, max_iter=1, gmres=0)
    assert rep["ir_iterations"] == 1, rep
    want = a.t() @ b  # the inverse is the transpose
    err = float((x.reshape(-1) - want).norm() / want.norm())
    assert np.isfinite(err) and err <= (10 * n * U32) ** 2 + 1e-13, err
