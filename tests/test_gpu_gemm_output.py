"""gemm without a C allocates one that is not cleared: every element has to be
written, whatever the memory held, also for an empty inner dimension."""
import pytest
import torch

import eigen_amd as ea

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 40, 3), (40, 1, 3), (17, 33, 0), (96, 80, 64),
                                   (129, 257, 5), (300, 200, 130), (700, 650, 40)])
@pytest.mark.parametrize("ta,tb", ["NN", "TT"])
def test_every_element_is_written(m, n, k, ta, tb):
    # the caching allocator hands the same block back: fill it with NaN first
    junk = torch.full((max(1, m * n),), float("nan"), dtype=torch.float64, device="cuda")
    del junk
    a = torch.ones((m, k) if ta == "N" else (k, m), dtype=torch.float64, device="cuda")
    b = torch.ones((k, n) if tb == "N" else (n, k), dtype=torch.float64, device="cuda")
    c = ea.gemm(a, b, transa=ta, transb=tb)
    assert c.shape == (m, n) and c.stride(0) == 1 and bool((c == k).all())
    assert bool((ea.gemm(a, b, alpha=0.0, transa=ta, transb=tb) == 0).all())
