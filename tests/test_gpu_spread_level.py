"""The rounding of the cells about the fine grid's centre, which every ray
crosses: as sums of hundreds of FP32 values one after the other it is a level
error of the PSF, and T x is off by that level.  T x of a disc with the FP32
operator against the FP64 one.

Tolerance 3e-7 relL2: a centre cell is summed 128 points at a time (rms rounding
of such a sum at most sqrt(128) 2^-24 / (2 sqrt 3) = 2e-7) and those sums in FP64;
1e-7 for the FP32 transforms."""

import numpy as np
import pytest

from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu


# grids with the centre inside a tile and on a tile's edge; items of the rule's
# size and far larger ones asked for
@pytest.mark.parametrize("n,P,chunk", [(1000, 720, None), (1454, 721, None),
                                       (900, 640, "4096"), (512, 400, "4096")])
def test_psf_level(torch_cuda, monkeypatch, n, P, chunk):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"PSF level n={n} P={P} chunk={chunk}")
    if chunk:
        monkeypatch.setenv("TOMOCAM_HIP_SPREAD_CHUNK", chunk)
    ang = (np.arange(P) * np.pi / P).astype(np.float32)
    r = torch.linspace(-1, 1, n, device="cuda", dtype=torch.float64)
    x = ((r[:, None] ** 2 + r[None, :] ** 2) < 0.6).double()[None].contiguous()
    ref = gpu.PointSpreadFunction64(ang.astype(np.float64), n).convolve(x)
    got = gpu.PointSpreadFunction(ang, n).convolve(x.float())
    assert rel_l2(got.cpu().numpy(), ref.cpu().numpy()) < 3e-7
