"""Toeplitz products at widths that no other test takes: the FP32-only plans of
2048 and 4096 points, and the widths whose smooth length has no plan near, which
take a plan of either kind (768, 2916, 5832 points) in FP32 alone.
Reference and tolerance (2e-5 relL2) as in test_gpu_toeplitz_plain.py; above 2000
the PSF comes from a geometry, as there."""

import numpy as np
import pytest

from conftest import rel_l2, announce
from test_gpu_toeplitz_plain import _psf, _ref

pytestmark = pytest.mark.gpu

# (n, S, M)
WIDTHS = [(1008, 2, 2048), (2025, 1, 4096), (330, 3, 768), (1310, 2, 2916),
          (2620, 1, 5832)]


@pytest.mark.parametrize("n,S,M", WIDTHS)
def test_width(torch_cuda, n, S, M):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"toeplitz width n={n} S={S} M={M}")
    if n < 2000:
        psf = gpu.PointSpreadFunction(psf_array=_psf(torch, n, n))
    else:
        psf = gpu.PointSpreadFunction(np.arange(40) * np.pi / 40, n)
    assert psf.fft_size == M
    g = torch.Generator(device="cuda").manual_seed(n + 1)
    x = torch.randn((S, n, n), device="cuda", generator=g)
    b = torch.randn((S, n, n), device="cuda", generator=g) * 1e-2
    ref = _ref(torch, x, psf.array())
    out, xtx = psf.convolve(x, with_dot=True)
    for s in range(S):
        assert rel_l2(out[s].cpu().numpy(), ref[s].cpu().numpy()) < 2e-5
    exact = float((x.double() * ref).sum())
    assert abs(xtx - exact) <= 1e-5 * float((x.double() * ref).abs().sum())
    grad = psf.gradient2(x, b)
    assert rel_l2(grad.cpu().numpy(), (ref - b.double()).cpu().numpy()) < 2e-5


@pytest.mark.parametrize("n", [330, 1310, 2620])
def test_mixed_form_refused(torch_cuda, n):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"toeplitz width n={n}: mixed form refused")
    psf = gpu.PointSpreadFunction(np.arange(5) * np.pi / 5, n)
    assert psf.tune(2, mixed=True) == 0
    with pytest.raises(ValueError, match="compile-time FFT plan"):
        psf.convolve_mixed(torch.zeros((1, n, n), device="cuda"))
