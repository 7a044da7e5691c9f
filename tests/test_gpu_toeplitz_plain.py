"""The FP32-only compile-time Toeplitz plans: one width per plan (the largest
it serves, so that no column of the padding is spare, or an odd one), against
the circulant product by torch's FP64 FFTs.  Tolerance 2e-5 relL2 (the bound
of the other Toeplitz tests)."""

import numpy as np
import pytest

from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu

# (n, S, M)
PLANS = [(243, 3, 486), (256, 2, 512), (287, 1, 576), (324, 4, 648),
         (432, 2, 864), (485, 3, 972), (512, 1, 1024), (576, 2, 1152),
         (647, 3, 1296), (768, 1, 1536), (863, 2, 1728), (972, 3, 1944),
         (1017, 2, 2250), (1296, 1, 2592), (1530, 2, 3072), (1727, 1, 3456),
         (1944, 2, 3888), (2590, 1, 5184), (3072, 1, 6144)]

# widths whose PSFs come from a geometry: a level PSF like the random one puts
# its mean into one row and one column of the FP32 spectrum, whose rounding
# reaches 2e-5 of the product at these widths on any FFT length (the
# runtime-plan kernels give 3.5e-5 at 4095)
LARGE = [(3455, 2, 6912), (3888, 1, 7776), (4095, 1, 8192)]


def _psf(torch, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    p = torch.rand((2 * n - 1, 2 * n - 1), device="cuda", generator=g)
    return (0.5 * (p + p.flip(0, 1))).contiguous()  # even


def _ref(torch, x, p):
    n = x.shape[-1]
    m = 1 << (2 * n - 1).bit_length()  # a few FFT sizes for all widths
    c = torch.zeros((m, m), device="cuda", dtype=torch.float64)
    i = (torch.arange(2 * n - 1, device="cuda") - (n - 1)) % m
    c[i[:, None], i[None, :]] = p.double()
    y = torch.fft.irfft2(torch.fft.rfft2(x.double(), s=(m, m))
                         * torch.fft.rfft2(c), s=(m, m))
    return y[:, :n, :n] / float(n) ** 3


@pytest.mark.parametrize("n,S,M", PLANS)
def test_plain_plan(torch_cuda, n, S, M):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"toeplitz plain plan n={n} S={S} M={M}")
    p = _psf(torch, n, n)
    psf = gpu.PointSpreadFunction(psf_array=p)
    assert psf.fft_size == M
    g = torch.Generator(device="cuda").manual_seed(n + 1)
    x = torch.randn((S, n, n), device="cuda", generator=g)
    b = torch.randn((S, n, n), device="cuda", generator=g) * 1e-2
    ref = _ref(torch, x, p)
    out, xtx = psf.convolve(x, with_dot=True)
    for s in range(S):
        assert rel_l2(out[s].cpu().numpy(), ref[s].cpu().numpy()) < 2e-5
    exact = float((x.double() * ref).sum())
    assert abs(xtx - exact) <= 1e-5 * float((x.double() * ref).abs().sum())
    grad = psf.gradient2(x, b)
    assert rel_l2(grad.cpu().numpy(), (ref - b.double()).cpu().numpy()) < 2e-5


@pytest.mark.parametrize("n,S,M", LARGE)
def test_plain_plan_large(torch_cuda, n, S, M):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"toeplitz plain plan n={n} S={S} M={M}")
    psf = gpu.PointSpreadFunction((np.arange(40) * np.pi / 40), n)
    assert psf.fft_size == M
    g = torch.Generator(device="cuda").manual_seed(n + 1)
    x = torch.randn((S, n, n), device="cuda", generator=g)
    ref = _ref(torch, x, psf.array())
    assert rel_l2(psf.convolve(x).cpu().numpy(), ref.cpu().numpy()) < 2e-5


@pytest.mark.parametrize("n", [250, 485])
def test_plain_plan_fused_commit(torch_cuda, monkeypatch, n):
    """run2 with the step committed inside the passes (y = sol, and after a
    rejection y = sol + beta (sol - x)) equals the separate commit kernel."""
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"toeplitz plain plan fused commit n={n}")
    p = _psf(torch, n, 5) * 100.0
    psf = gpu.PointSpreadFunction(psf_array=p)
    g = torch.Generator(device="cuda").manual_seed(n)
    x0 = torch.rand((3, n, n), device="cuda", generator=g)
    b = psf.convolve(torch.rand((3, n, n), device="cuda", generator=g))
    res = []
    for fused in ("1", "0"):
        monkeypatch.setenv("TOMOCAM_HIP_FUSED_COMMIT", fused)
        out, err, xerr, st = gpu.run2(psf, x0, b, 6, 6.0, 1e4,
                                      sino_sq=float((b * b).sum()) * 100)
        res.append((out.cpu().numpy(), st))
    assert res[0][1]["attempts"] == res[1][1]["attempts"]
    assert np.array_equal(res[0][0], res[1][0])


def test_plain_plan_has_no_mixed_form(torch_cuda):
    torch = torch_cuda
    from tomocam_amd import gpu
    psf = gpu.PointSpreadFunction(psf_array=_psf(torch, 250, 1))
    announce("toeplitz plain plan: mixed form refused")
    assert psf.tune(4, mixed=True) == 0
    with pytest.raises(ValueError, match="compile-time FFT plan"):
        psf.convolve_mixed(torch.zeros((1, 250, 250), device="cuda"))
