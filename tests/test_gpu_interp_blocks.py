"""Interpolation from the blocked half grid: footprints inside the stored
columns are read block by block, those that reach past column 0 or nf/2 cell by
cell; rays along and close to the grid's axes mix both in one wave.

Reference: the FP64 oracle's exact NUDFT, tolerance 1e-5 relL2 per slice (the
bound of the projector tests: kernel error 1.4e-7, FP32 rounding below 1e-6).
A slice's result does not depend on the slices beside it."""

import numpy as np
import pytest

from oracle import tomocam_oracle as O
from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu


# grids of 46 (few columns), 128 and 400 points, with and without a line plan;
# one slice, part of a chunk of eight, a whole one, and whole ones with a rest
@pytest.mark.parametrize("N,S", [(23, 1), (64, 7), (64, 8), (200, 17)])
def test_projection_near_the_axes(torch_cuda, N, S):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"interpolation near the axes N={N} S={S}")
    off = np.array([0.0, 1e-4, -1e-4, 0.01, -0.01, 4.0 / N, -4.0 / N])
    ang = np.concatenate([c + off for c in
                          (-np.pi / 2, 0.0, np.pi / 4, np.pi / 2, np.pi)])
    ang = ang.astype(np.float32)
    rng = np.random.default_rng(N + S)
    x = rng.random((S, N, N)).astype(np.float32)
    xd = torch.from_numpy(x).cuda()
    got = gpu.project(xd, ang)
    ref = O.project(x, ang.astype(np.float64), exact=True)
    for g, r in zip(got.cpu().numpy(), ref):
        assert rel_l2(g, r) < 1e-5
    for s in {0, S - 1}:
        assert torch.equal(gpu.project(xd[s:s + 1], ang)[0], got[s])
