"""The look-ahead factorization's interchanges and U rows at widths where the
kernel's sixteen columns a wave, 16-row blocks and 128-row panels end, with
16-byte rows and without.

The matrix is a row-permuted Householder reflection (condition 1): the FP16
hi/lo split keeps 22 bits, so with a factor of relative error e0 <= 10 n 2^-22
(ten for the elimination's growth) the solution after one refinement step is
off by at most e0^2 and the FP64 residual's 1e-13.  A row or a column in the
wrong place makes e0 of order one."""
import numpy as np
import pytest
import torch

from eigen_amd import mixed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [129, 130, 143, 144, 145, 159, 160, 255, 256, 257, 272, 300, 385, 400,
                               513, 1000, 1297])
def test_one_refinement_step(n):
    print(f"n={n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    v = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    perm = torch.randperm(n, device="cuda", generator=g)
    a = torch.eye(n, dtype=torch.float64, device="cuda")[perm]
    a -= (2.0 / (v @ v)) * torch.outer(v[perm], v)
    b = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    a = a.t().contiguous().t()
    x, rep = mixed.gesv_ir(a, b, precision="fp16x3", check_converged=False, max_iter=1, gmres=0)
    assert rep["ir_iterations"] == 1, rep
    want = a.t() @ b  # the inverse is the transpose
    err = float((x.reshape(-1) - want).norm() / want.norm())
    assert np.isfinite(err) and err <= (10 * n * 2.0 ** -22) ** 2 + 1e-13, err
