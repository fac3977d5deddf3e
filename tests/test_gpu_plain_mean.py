"""The plain mean of DP where a uniform x2 has no cosine transform (N/2 with a factor 7 or more): DIRECT leaves it at
zero (direct.f:894-898), so the solution agrees with the long-double oracle mean included, at the suite's 1e-12. The
dense transform alone, as matrix products, and in a one-launch batch."""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import interior

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(24, 14, 10), (40, 74, 8), (150, 22, 6), (160, 134, 4)])
def test_plain_mean_without_cosine_transform(torch_cuda, m, n, l):
    g = grid.make_grid(m, n, l, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m + n)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = interior(oracle.direct(g, rhs, extended=True))

    def check(what, d):
        torch_cuda.cuda.synchronize()
        got = interior(eddyproj.to_host(d))
        err = np.abs(got - ref).max() / np.abs(ref).max()
        print("plain mean", m, n, l, what, "%.1e mean %.1e" % (err, got.mean() / np.abs(ref).max()), flush=True)
        assert err <= 1e-12

    plan = eddyproj.Plan(g)
    for timing in (False, True):  # the fused plane kernel where the plan takes it, and the separate ones
        plan.enable_timing(timing)
        check("plan", plan.direct(eddyproj.to_device(rhs)))
    plan.close()
    d = eddyproj.to_device(rhs)
    b = eddyproj.Batch([g])
    b.set_mode(eddyproj.BATCH_QUEUES)
    b.bind([d])
    b.direct()
    check("batch", d)
    b.close()
