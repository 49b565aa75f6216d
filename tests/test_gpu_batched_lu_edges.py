"""The batched LU's FP32 factor and solves at the edges of their blocks: 16-row
tiles and panels, 64-row diagonal blocks, the size classes' ends, four and five
right-hand sides.

The systems are row-permuted Householder reflections, condition 1: with an FP32
factor of relative error e0 <= 10 n u32 (a factor of ten for the growth of the
elimination) each refinement step multiplies the error by at most e0, so three
steps reach 1e-14 at n = 256 from the FP32 factor.  A wrong entry anywhere in
the factor or the solves makes e0 of order one: the refinement stalls and the
system falls to the FP64 refactor (info 1) or needs more steps."""
import numpy as np
import pytest
import torch

from eigen_amd import batched
from tests import inputs

pytestmark = pytest.mark.gpu
EDGES = [1, 2, 3, 4, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 95, 127, 128, 129,
         143, 144, 145, 191, 192, 193, 207, 208, 209, 239, 240, 241, 254, 255, 256]


@pytest.mark.parametrize("nrhs", [1, 4, 5, 8])
def test_edges_refine_from_the_fp32_factor(nrhs):
    n = np.array(EDGES * 3, dtype=np.int32)
    offA = np.concatenate([[0], np.cumsum(n.astype(np.int64) ** 2)[:-1]])
    offB = np.concatenate([[0], np.cumsum(n.astype(np.int64) * nrhs)[:-1]])
    A, B, X = [], [], []
    for i, k in enumerate(n):
        g = inputs.rng(5000 + 131 * i + nrhs)
        v = g.standard_normal(k)
        a = (np.eye(k) - 2.0 * np.outer(v, v) / (v @ v))[g.permutation(k)]
        x = g.standard_normal((k, nrhs))
        A.append(a.ravel(order="F"))
        B.append((a @ x).ravel(order="F"))
        X.append(x.ravel(order="F"))
    A, B, X = map(np.concatenate, (A, B, X))
    dev = [torch.from_numpy(np.ascontiguousarray(t)).cuda() for t in (offA, n, A, offB, B)]
    got, info, iters = batched.dgesv_ir_batched(*dev[:4], nrhs, dev[4])
    got, info, iters = got.cpu().numpy(), info.cpu().numpy(), iters.cpu().numpy()
    for i, k in enumerate(n):
        sl = slice(offB[i], offB[i] + k * nrhs)
        err = np.linalg.norm(got[sl] - X[sl]) / np.linalg.norm(X[sl])
        assert info[i] == 0 and iters[i] <= 3, (k, info[i], iters[i], err)
        # backward error 1e-14 in the infinity norms, condition <= n there
        assert err <= 4e-14 * k, (k, err)
