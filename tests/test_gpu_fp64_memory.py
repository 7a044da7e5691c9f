"""What an FP64 projector call leaves cached: its buffers, so that a repeated call
allocates nothing, but not the grids of a whole stack (about 2 GB of grid and
samples at a time, and the spreading's scratch of at most 1 GB).  The results do
not depend on how the stack is split."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


# 72 slices: 4.6 GB of grids and samples
@pytest.mark.parametrize("N,S", [(200, 2), (1000, 72)])
def test_cached_buffers(torch_cuda, N, S):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"FP64 projectors, cached memory: N={N} S={S}")
    ang = np.arange(9) * (np.pi / 9)
    x = torch.rand((S, N, N), device="cuda", dtype=torch.float64)

    def calls(x):
        y = gpu.project(x, ang)
        return y, gpu.backproject(y, ang), gpu.gradient(x, x, ang)

    first = calls(x)
    gpu.release_cached()
    assert all(torch.equal(a, b) for a, b in zip(calls(x), first))
    mallocs, _, cached = gpu.alloc_stats()
    assert cached < 3.2e9
    assert all(torch.equal(a, b) for a, b in zip(calls(x), first))
    assert gpu.alloc_stats()[0] == mallocs
    for s in (0, S // 2, S - 1):
        assert all(torch.equal(a[0], b[s])
                   for a, b in zip(calls(x[s:s + 1]), first))
    gpu.release_cached()
