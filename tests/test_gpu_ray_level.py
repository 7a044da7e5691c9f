"""The level taken off a ray before the ramp filter does not follow single
pixels: a hot pixel where the level is sampled costs no more accuracy than one
beside it.  FBP against the FP64 form; the two errors are of one kind and size,
so the bound is 1.5 times (the mean of the samples gave several times)."""

import numpy as np
import pytest

from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu


# planned ray length (direct transform), chirp on a planned length, and the
# runtime-plan kernels
@pytest.mark.parametrize("N,runtime", [(1536, False), (1531, False),
                                       (1531, True)])
def test_hot_pixel_at_a_level_sample(torch_cuda, monkeypatch, N, runtime):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"ray level N={N} runtime={runtime}")
    if runtime:
        monkeypatch.setenv("TOMOCAM_HIP_CT_LINES", "0")
    P = 5
    ang = (np.arange(P) * np.pi / P).astype(np.float32)
    t = np.linspace(-1, 1, N)
    base = np.sqrt(np.maximum(0.7 - t * t, 0.0)) + 0.05
    base = base + 0.01 * np.random.default_rng(N).random((1, P, N))

    def err(k, up):
        y = base.copy()
        y[:, :, k] += up
        y32 = torch.from_numpy(y.astype(np.float32)).cuda()
        got = gpu.backproject(y32, ang, fbp=True)
        ref = gpu.backproject(y32.double(), ang.astype(np.float64), fbp=True)
        return rel_l2(got.cpu().numpy(), ref.cpu().numpy())

    for k in (1, 4, 7):
        at = (2 * k + 1) * N // 16
        for up in (1e4, -1e4):
            assert err(at, up) < 1.5 * err(at + 5, up)
