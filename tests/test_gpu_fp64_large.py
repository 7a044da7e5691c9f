"""FP64 projectors at sizes that take more than one launch: more sample points
than 2^32 threads, sixteen a point, hold (a larger launch runs in part, without an
error), and more slices than the spreading takes at once.  A slice and a ray are computed alike in any call, so parts of the
results equal those of small calls bit for bit."""

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


# 2^28 points and some, in many slices and in one
@pytest.mark.parametrize("S,N,P", [(256, 16, 65600), (1, 64, (1 << 22) + 64)])
def test_many_points(torch_cuda, S, N, P):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"FP64 project S={S} N={N} P={P}")
    ang = np.arange(P) * (np.pi / P)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((S, N, N), device="cuda", generator=g, dtype=torch.float64)
    got = gpu.project(x, ang)
    pick = [0, 1, P // 2, P - 2, P - 1]
    for s in sorted({0, S // 2 - 1, S // 2, S - 1} & set(range(S))):
        ref = gpu.project(x[s:s + 1], ang[pick])
        assert torch.equal(got[s, pick], ref[0])
    del got
    gpu.release_cached()


def test_many_slices(torch_cuda):
    torch = torch_cuda
    from tomocam_amd import gpu
    S, N, P = 4 * 65535 + 9, 2, 2
    announce(f"FP64 backproject S={S} N={N} P={P}")
    ang = np.array([0.1, 1.2])
    g = torch.Generator(device="cuda").manual_seed(2)
    y = torch.rand((S, P, N), device="cuda", generator=g, dtype=torch.float64)
    got = gpu.backproject(y, ang)
    for s in (0, 65535, 4 * 65535 - 1, 4 * 65535, S - 1):
        assert torch.equal(got[s], gpu.backproject(y[s:s + 1], ang)[0])
    del got
    gpu.release_cached()
