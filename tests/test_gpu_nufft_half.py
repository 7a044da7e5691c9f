"""The half-grid NUFFT path at the sizes where it can go wrong: real rows and
rays are transformed in pairs, only columns 0 .. nf/2 of the fine grid are
kept, an even ray's end sample is split over both ends, and a spreading
workgroup takes 2, 4 or 8 slices.

Reference: the FP64 oracle's exact NUDFT.  Tolerance 1e-5 relL2 per slice, the
bound of the projector tests (the kernel's own error is 1.4e-7 and FP32
rounding of a few transforms stays below 1e-6; the ramp amplifies it by up to
the ratio of the sinogram's norm to the filtered one's, below 10 here)."""

import numpy as np
import pytest

from oracle import tomocam_oracle as O
from tomocam_amd import phantom as PH
from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu

# (N, P, S): smallest widths, odd and even, odd and even pair counts, planned
# ray lengths (64, 96, 128), grids on and off a tile edge (nf/2 + 1 = 33, 65),
# slice groups of 1 .. 9
SHAPES = [(2, 1, 1), (3, 2, 2), (5, 3, 3), (8, 5, 1), (16, 4, 5), (31, 7, 4),
          (32, 17, 2), (33, 1, 9), (64, 9, 3), (65, 12, 8), (96, 5, 1),
          (101, 6, 2), (128, 3, 7)]


def _angles(P, kind):
    a = PH.angles(P)
    if kind == "axes":  # rays on the grid axes and in all four quadrants
        a = (np.arange(P) * np.pi / 2 - np.pi).astype(np.float32)
    return a


def _check(got, ref):
    for g, r in zip(got, ref):
        assert rel_l2(g, r) < 1e-5


@pytest.mark.parametrize("runtime", [False, True])
@pytest.mark.parametrize("kind", ["uniform", "axes"])
@pytest.mark.parametrize("N,P,S", SHAPES)
def test_projectors_at_edge_sizes(torch_cuda, monkeypatch, N, P, S, kind,
                                  runtime):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"half-grid projectors N={N} P={P} S={S} {kind} rt={runtime}")
    if runtime:
        monkeypatch.setenv("TOMOCAM_HIP_CT_LINES", "0")
    ang = _angles(P, kind)
    a64 = ang.astype(np.float64)
    rng = np.random.default_rng(100 * N + P)
    # slices of very different level: no slice may reach into another
    lev = 10.0 ** (3.0 * (np.arange(S) % 3) - 3.0)
    x = (rng.random((S, N, N)) * lev[:, None, None]).astype(np.float32)
    y = (rng.random((S, P, N)) * lev[:, None, None]).astype(np.float32)
    xd, yd = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    _check(gpu.project(xd, ang).cpu().numpy(), O.project(x, a64, exact=True))
    _check(gpu.backproject(yd, ang).cpu().numpy(),
           O.backproject(y, a64, exact=True))
    if N >= 16:
        _check(gpu.backproject(yd, ang, fbp=True).cpu().numpy(),
               O.backproject(y, a64, fbp=True, exact=True))
    g = gpu.gradient(xd, torch.zeros_like(xd), ang).cpu().numpy()
    _check(g, O.gradient_nufft(x, 0.0, a64, exact=True))


def test_slices_do_not_mix(torch_cuda):
    """A slice of NaN leaves its neighbours' results as they are."""
    torch = torch_cuda
    from tomocam_amd import gpu
    announce("half-grid projectors: NaN slice")
    N, P, S = 40, 15, 6
    ang = PH.angles(P)
    g = torch.Generator(device="cuda").manual_seed(3)
    for fn, shape in ((gpu.project, (S, N, N)), (gpu.backproject, (S, P, N))):
        a = torch.rand(shape, device="cuda", generator=g)
        ref = fn(a, ang)
        a[2] = float("nan")
        got = fn(a, ang)
        keep = [0, 1, 3, 4, 5]
        assert torch.equal(got[keep], ref[keep])
        assert torch.isnan(got[2]).all()


@pytest.mark.parametrize("N", [5900, 8001])
def test_lines_too_long_for_two_buffers(torch_cuda, N):
    """Grid and ray lengths above the two-buffer limit: single samples of the
    exact sums, and the adjoint identity, which holds to the sums' rounding."""
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"long lines N={N}")
    P = 3
    ang = PH.angles(P)
    g = torch.Generator(device="cuda").manual_seed(N)
    x = torch.rand((1, N, N), device="cuda", generator=g)
    y = torch.rand((1, P, N), device="cuda", generator=g)
    px, pty = gpu.project(x, ang).double(), gpu.backproject(y, ang).double()
    a, b = float((px * y.double()).sum()), float((x.double() * pty).sum())
    assert abs(a - b) <= 2e-6 * abs(a)
    # P^T y at a few pixels: Re sum_j V_j e^{i(k1 x_j + k2 y_j)} / N^2
    V = O.centered_ray_dft(y[0].double().cpu().numpy().astype(complex), -1)
    gx, gy = O.polar_grid(ang.astype(np.float64), N)
    scale = float(pty.abs().max())
    for k2, k1 in ((0, 0), (N // 2, N // 2), (N - 1, 7), (17, N - 1)):
        ref = np.real(np.sum(V * np.exp(1j * ((k1 - N // 2) * gx
                                              + (k2 - N // 2) * gy)))) / N ** 2
        assert abs(float(pty[0, k2, k1]) - ref) <= 1e-5 * scale
