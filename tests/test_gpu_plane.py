"""The fused plane kernels (x2 transform, line solves, inverse transform of a y-mode in one workgroup):
planes of the cosine and of the dense form at their edges, against the three separate kernels (which run
while kernel timing is on) and against the long-double oracle at the suite's 1e-12.
"""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import interior, rel_maxdiff_nomean

pytestmark = pytest.mark.gpu

# (m, n, l, z_beta): cosine: N = 4 (one butterfly), N/2 odd (5), 3-5-smooth, 64, 128, 256; M = 3, ragged, the
# largest plane of L >= 128; dense: odd N, N past a 16-block, M past 16 and 112 lines, 127 x 127
SHAPES = [(3, 4, 6, None), (17, 10, 8, None), (33, 30, 12, None), (64, 64, 8, None), (128, 128, 128, None),
          (61, 128, 130, None), (20, 256, 128, None), (16, 150, 8, None), (5, 7, 6, None), (16, 16, 12, 1.2),
          (33, 17, 10, 1.2), (113, 33, 6, None), (127, 127, 6, 1.3), (40, 100, 8, 1.1)]


@pytest.mark.parametrize("m,n,l,zb", SHAPES)
def test_plane_direct(torch_cuda, m, n, l, zb):
    g = grid.make_grid(m, n, l, x_beta=1.4, z_beta=zb)
    u, v, w = configs.random_uniform_velocity(g, m + n)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    tol = max(1e-12, 4 * rel_maxdiff_nomean(oracle.direct(g, rhs), ref))
    plan = eddyproj.Plan(g)
    got = []
    for timing in (False, True):
        plan.enable_timing(timing)
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        torch_cuda.cuda.synchronize()
        got.append(eddyproj.to_host(d))
        err = rel_maxdiff_nomean(got[-1], ref)
        print("plane", m, n, l, zb, "separate" if timing else "plan", "%.2e" % err, flush=True)
        assert err <= tol
    # the same algorithm in the same precision: the plain mean included
    assert np.abs(got[0] - got[1]).max() <= 1e-12 * np.abs(got[1]).max()
    plan.enable_timing(False)
    d = eddyproj.to_device(rhs)
    plan.direct_refined(d, sweeps=3)
    phi = eddyproj.to_host(d)
    b = interior(rhs)
    assert np.linalg.norm(b - interior(oracle.laplacian(g, phi))) <= 1e-10 * np.linalg.norm(b)
    plan.close()


@pytest.mark.parametrize("zb", [None, 1.2])
def test_plane_projection_removes_mean(torch_cuda, zb):
    """The zero mode's shift and mean correction: an RHS whose volume-weighted mean is not zero."""
    g = grid.make_grid(40, 24, 16, x_beta=1.4, z_beta=zb)
    u, v, w = configs.random_uniform_velocity(g, 9)
    dps = []
    for timing in (False, True):
        plan = eddyproj.Plan(g)
        plan.enable_timing(timing)
        t = [eddyproj.to_device(a) for a in (u, v, w)]
        o = [a.clone() for a in t]
        dp = torch_cuda.zeros_like(t[0])
        plan.project(*t, *o, dp, configs.DT)
        torch_cuda.cuda.synchronize()
        dps.append(eddyproj.to_host(dp))
        plan.close()
    ref = oracle.direct(g, configs.rhs_from_velocity(g, u, v, w), extended=True)
    assert rel_maxdiff_nomean(dps[0], ref) <= 1e-12
    assert np.abs(dps[0] - dps[1]).max() <= 1e-12 * np.abs(dps[1]).max()
