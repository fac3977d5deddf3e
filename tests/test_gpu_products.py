"""The FP64 matrix products of a stretched or odd x2 over their tiles: contractions of every length mod 8,
tiles cut by C's edges, odd leading dimensions with many modes (64 x 64 tiles from registers), even ones
(the LDS-staged tiles) and 32 x 64 tiles; the zero mode's shift and mean included. Against the long-double
oracle at the suite's 1e-12 or four times the FP64 oracle's own error.
"""
import os

import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu

SHAPES = [(140, 129, 6), (135, 130, 6), (150, 131, 4), (133, 132, 6), (134, 133, 4), (33, 134, 8), (6, 135, 6),
          (47, 136, 4), (67, 131, 342), (66, 130, 342), (128, 128, 256)]


@pytest.mark.parametrize("m,n,l", SHAPES)
def test_products(torch_cuda, m, n, l):
    oracle.set_threads(min(16, os.cpu_count() or 1))
    g = grid.make_grid(m, n, l, x_beta=1.4, z_beta=1.1)
    u, v, w = configs.random_uniform_velocity(g, m + n)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    tol = max(1e-12, 4 * rel_maxdiff_nomean(oracle.direct(g, rhs), ref))
    for form in (1, 2):
        plan = eddyproj.Plan(g, tuning={"zgemm": form})
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        t = [eddyproj.to_device(a) for a in (u, v, w)]
        o = [a.clone() for a in t]
        dp = torch_cuda.zeros_like(t[0])
        plan.project(*t, *o, dp, configs.DT)
        torch_cuda.cuda.synchronize()
        errs = [rel_maxdiff_nomean(eddyproj.to_host(a), ref) for a in (d, dp)]
        phi = eddyproj.to_host(dp)[1:-1, 1:-1, 1:-1]
        print("products", m, n, l, form, ["%.2e" % e for e in errs], flush=True)
        assert max(errs) <= tol
        assert abs(phi.mean()) <= 1e-11 * np.abs(phi).max()
        plan.close()
