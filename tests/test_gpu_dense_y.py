"""Periodic lengths that the radix FFT does not take (odd L, or L/2 with a prime factor >= 7): the
dense real DFT of the y transforms, at the edges of its 16-output blocks and 4-sample steps, of
its 16-pencil groups and of the LDS (narrower tiles), against the long-double oracle.

Tolerance: the suite's 1e-12 on DIRECT. A DFT sum of L terms in FP64 is within L eps ~ 3e-13 of
exact in the worst case at L = 1502, and sqrt(L) eps ~ 1e-14 for terms of random sign.
"""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu

# (m, n, l): l = 7 (one step, one block), 29..33 (L/2 = 14, 15, 16: the block edge), 62 (L/2 = 31),
# 112, 127, 203; 1502 narrows the tile to 8 pencils; m below, at and past 16-pencil groups
SHAPES = [(5, 4, 7), (16, 6, 29), (17, 4, 31), (33, 4, 33), (12, 8, 62), (65, 6, 112), (40, 5, 127), (9, 4, 203),
          (6, 4, 1502)]


def _problem(m, n, l, seed, **kw):
    g = grid.make_grid(m, n, l, x_beta=1.5, **kw)
    u, v, w = configs.random_uniform_velocity(g, seed)
    return g, (u, v, w), configs.rhs_from_velocity(g, u, v, w)


@pytest.mark.parametrize("m,n,l", SHAPES)
def test_dense_y_direct(torch_cuda, m, n, l):
    g, _, rhs = _problem(m, n, l, l)
    ref = oracle.direct(g, rhs, extended=True)
    for tun in (None, {"yfft_pencils": 4}, {"yfft_pencils": 64}):
        plan = eddyproj.Plan(g, tuning=tun)
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        torch_cuda.cuda.synchronize()
        err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
        print("dense y", m, n, l, tun, "%.2e" % err, flush=True)
        assert err <= 1e-12
        plan.close()


@pytest.mark.parametrize("cyl", [False, True])
@pytest.mark.parametrize("precision,sweeps,tol", [(eddyproj.EDDY_FP64, 0, 1e-12), (eddyproj.EDDY_FP32_REFINE, 3, 1e-10)])
def test_dense_y_projection(torch_cuda, cyl, precision, sweeps, tol):
    """The fused divergence and the residual and update forms (FP32: 3 sweeps, the suite's 1e-10)."""
    g, (u, v, w), rhs = _problem(21, 8, 62, 3, cyl=cyl)
    ref = oracle.direct(g, rhs, extended=True)
    t = [eddyproj.to_device(a) for a in (u, v, w)]
    o = [a.clone() for a in t]
    dp = torch_cuda.zeros_like(t[0])
    plan = eddyproj.Plan(g)
    plan.project(*t, *o, dp, configs.DT, precision=precision, sweeps=sweeps)
    torch_cuda.cuda.synchronize()
    phi = eddyproj.to_host(dp)
    assert rel_maxdiff_nomean(phi, ref) <= tol
    np.testing.assert_array_equal(phi[:, 0, 1:-1], phi[:, -2, 1:-1])
    np.testing.assert_array_equal(phi[:, -1, 1:-1], phi[:, 1, 1:-1])
    plan.close()
