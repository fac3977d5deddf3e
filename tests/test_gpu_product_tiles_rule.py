"""FP64 products whose row tiles four waves do not divide, on the side of the rule where a batch's tiles go four to
a workgroup (the last of two rounds of waves 0.55 to 0.85 full): remainders of one, two, three and none, x-major
and p-major operands, odd and even leading dimensions, the zero mode included. Against the long-double oracle at
the suite's 1e-12 or four times the FP64 oracle's own error."""
import os

import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


# 25, 30, 15 and 20 tiles a batch
@pytest.mark.parametrize("m,n,l", [(135, 131, 70), (163, 129, 60), (135, 90, 120), (146, 122, 90)])
def test_tiles_four_to_a_workgroup(torch_cuda, m, n, l):
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
        print("tiles, four to a workgroup", m, n, l, form, ["%.2e" % e for e in errs], "%.1e" % tol, flush=True)
        assert max(errs) <= tol
        plan.close()
