"""Plans on either side of each line of the fused plane kernel's rule (plane size, periodic length, radix), in FP64 and
FP32: the plan's solution against the three separate kernels, which run while kernel timing is on, and the small ones
against the long-double oracle at the suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu

# (m, n, l, whether the plan takes the plane kernel): planes of 3072 and 3136; 4096 at L = 90 and 96; 6144 and 6208
# past L = 256; 8192 at 120, 144, 256 and 270; the largest, 16384; N/2 = 30 with a radix of 2; N = 4
SHAPES = [(48, 64, 6, True), (49, 64, 6, False), (64, 64, 90, False), (64, 64, 96, True), (96, 64, 270, True),
          (97, 64, 270, False), (64, 128, 120, False), (64, 128, 144, True), (128, 64, 256, True),
          (128, 64, 270, False), (128, 128, 240, True), (60, 60, 160, False), (51, 60, 128, True), (800, 4, 60, False)]


@pytest.mark.parametrize("m,n,l,fused", SHAPES)
def test_plane_rule(torch_cuda, m, n, l, fused):
    g = grid.make_grid(m, n, l, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m + l)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    plan = eddyproj.Plan(g)
    got = {}
    for timing in (False, True):
        plan.enable_timing(timing)
        got[timing] = []
        for solve in (plan.direct, lambda d: plan.direct_refined(d, 4, residual=False)):
            d = eddyproj.to_device(rhs)
            solve(d)
            torch_cuda.cuda.synchronize()
            got[timing].append(eddyproj.to_host(d))
    plan.close()
    errs = [rel_maxdiff_nomean(a, b) for a, b in zip(got[False], got[True])]
    if m * n * l <= 400000:
        errs.append(rel_maxdiff_nomean(got[False][0], oracle.direct(g, rhs, extended=True)))
    print("plane rule", m, n, l, ["%.1e" % e for e in errs], flush=True)
    assert max(errs) <= 1e-12
    # the three kernels round alike every time, the fused one in its own way
    assert (max(errs[:2]) > 0) == fused
