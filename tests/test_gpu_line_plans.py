"""Ray transforms on every compile-time line plan, as the sources list them: rays
of the planned length itself (both directions) and rays whose chirp takes the
length (backprojection, plain and with the ramp), an odd number of rays a slice
and more lines than one workgroup holds.

Each result against the same call on the runtime-plan kernels, which the
exact-NUDFT projector tests pin: relL2 <= 2e-6 as in test_gpu_fft_lines.py (two
FP32 FFT orderings), twice that behind the ramp, which weights the rounding of
the high frequencies by up to sqrt(3) times its mean."""

import os
import re

import pytest

from tomocam_amd import phantom as PH
from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu

with open(os.path.join(os.path.dirname(__file__), "..", "tomocam_amd", "csrc",
                       "fft_lines_ct.h")) as _f:
    LENGTHS = sorted(int(v) for v in re.findall(r"using L(\d+) =", _f.read()))


def _chirp_width(L):
    """The largest width that has no plan of its own and whose chirp takes L."""
    below = max([0] + [m for m in LENGTHS if m < L])
    for N in (L // 2, L // 2 - 1):
        if N not in LENGTHS and 2 * N - 1 > below:
            return N
    raise AssertionError(L)


@pytest.mark.parametrize("L", LENGTHS)
def test_ray_transforms(torch_cuda, monkeypatch, L):
    torch = torch_cuda
    from tomocam_amd import gpu
    S, P = (20, 3) if L < 700 else (4, 3) if L < 2000 else (1, 5)
    ang = PH.angles(P)
    g = torch.Generator(device="cuda").manual_seed(L)

    def both(fn, tol):
        monkeypatch.delenv("TOMOCAM_HIP_CT_LINES", raising=False)
        a = fn()
        monkeypatch.setenv("TOMOCAM_HIP_CT_LINES", "0")
        b = fn()
        for s in range(S):
            assert rel_l2(a[s].cpu().numpy(), b[s].cpu().numpy()) <= tol

    # the grid of twice the width has to fit as well
    widths = ([L] if 2 * L <= LENGTHS[-1] else []) + [_chirp_width(L)]
    for N in widths:
        announce(f"line plan {L}: rays of {N} samples, {S} x {P}")
        y = torch.rand((S, P, N), device="cuda", generator=g)
        both(lambda: gpu.backproject(y, ang), 2e-6)
        both(lambda: gpu.backproject(y, ang, fbp=True), 4e-6)
        if N == L:
            x = torch.rand((S, N, N), device="cuda", generator=g)
            both(lambda: gpu.project(x, ang), 2e-6)


def test_list_is_complete():
    assert len(LENGTHS) == 45
