"""FP64 products whose row tiles four waves do not divide, the tiles of a batch taken four at a time: whole
fours, a remainder of one and of two, odd and even leading dimensions, the zero mode included. Against the
long-double oracle at the suite's 1e-12 or four times the FP64 oracle's own error."""
import os

import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(135, 131, 54), (144, 150, 54), (163, 129, 50), (168, 190, 36), (144, 246, 50)])
def test_product_tiles(torch_cuda, m, n, l):
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
        dp = torch_cuda.zeros_like(t[0])
        plan.project(*t, *[a.clone() for a in t], dp, configs.DT)
        torch_cuda.cuda.synchronize()
        errs = [rel_maxdiff_nomean(eddyproj.to_host(a), ref) for a in (d, dp)]
        print("product tiles", m, n, l, form, ["%.2e" % e for e in errs], flush=True)
        assert max(errs) <= tol
        plan.close()
