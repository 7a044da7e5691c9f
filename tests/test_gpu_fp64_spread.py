"""The FP64 tile-owned spreading and the sixteen-lane gather at the sizes where
they can go wrong: grids of one tile and of partial tiles, one to five slices
(groups of 2 and 4), batches of points that end inside a ray, angles on the
axes, more than 2048 angles.  Reference: the oracle's exact NUDFT; bound 1e-10
relL2 as for the other FP64 operators.  Results repeat bit for bit."""

import numpy as np
import pytest

from oracle import tomocam_oracle as O
from conftest import rel_l2, announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,S", [(2, 1, 1), (5, 3, 2), (16, 9, 3),
                                   (17, 30, 4), (40, 33, 5), (33, 2100, 1)])
def test_fp64_projectors_at_edge_sizes(torch_cuda, N, P, S):
    torch = torch_cuda
    from tomocam_amd import gpu
    announce(f"FP64 projectors N={N} P={P} S={S}")
    rng = np.random.default_rng(N + P)
    ang = np.arange(P) * (np.pi / 2 if P < 10 else np.pi / P) - 0.5 * np.pi
    x = rng.standard_normal((S, N, N))
    y = rng.standard_normal((S, P, N))
    xd, yd = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    b = gpu.backproject(yd, ang)
    for got, ref in ((gpu.project(xd, ang), O.project(x, ang, exact=True)),
                     (b, O.backproject(y, ang, exact=True)),
                     (gpu.gradient(xd, torch.zeros_like(xd), ang),
                      O.gradient_nufft(x, 0.0, ang, exact=True))):
        for s in range(S):
            assert rel_l2(got[s].cpu().numpy(), ref[s]) < 1e-10
    assert torch.equal(b, gpu.backproject(yd, ang))


def test_fp64_plans_shared_by_threads_and_streams(torch_cuda):
    """More geometries than the plan cache keeps, from two threads on streams
    of their own: every result equals the single-threaded one."""
    import threading
    torch = torch_cuda
    from tomocam_amd import gpu
    announce("FP64 plans: two threads, 20 geometries")
    rng = np.random.default_rng(5)
    jobs = []
    for k in range(20):
        P, N = 5 + k, 20 + k
        jobs.append((torch.from_numpy(rng.standard_normal((2, P, N))).cuda(),
                     np.arange(P) * np.pi / P))
    ref = [gpu.backproject(y, a) for y, a in jobs]
    torch.cuda.synchronize()
    out = [[None] * len(jobs) for _ in range(2)]
    errs = []

    def run(t):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                order = range(len(jobs)) if t == 0 else reversed(range(len(jobs)))
                for k in order:
                    out[t][k] = gpu.backproject(*jobs[k])
            st.synchronize()
        except Exception as e:  # reported below
            errs.append(e)

    th = [threading.Thread(target=run, args=(t,)) for t in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errs, errs
    for t in range(2):
        for k in range(len(jobs)):
            assert torch.equal(out[t][k], ref[k])
