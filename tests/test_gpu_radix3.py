"""Transform lengths 3 * 2^k with passes of their own (half-lengths 24, 48, 96, 192) along y and x2, whole and
ragged tiles and batches, against the long-double oracle at the suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(20, 4, 48), (33, 6, 96), (17, 4, 192), (9, 4, 384), (20, 48, 4), (140, 96, 6),
                                   (33, 192, 4), (20, 384, 4), (130, 192, 96)])
def test_radix3_lengths(torch_cuda, m, n, l):
    g = grid.make_grid(m, n, l, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m + n + l)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    plan = eddyproj.Plan(g)
    for timing in (False, True):  # the fused plane kernel where the plan takes it, and the separate ones
        plan.enable_timing(timing)
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        torch_cuda.cuda.synchronize()
        err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
        print("radix 3", m, n, l, "%.2e" % err, flush=True)
        assert err <= 1e-12
    b = eddyproj.Batch([g])
    b.set_mode(eddyproj.BATCH_QUEUES)
    d = eddyproj.to_device(rhs)
    b.bind([d])
    b.direct()
    torch_cuda.cuda.synchronize()
    assert rel_maxdiff_nomean(eddyproj.to_host(d), ref) <= 1e-12
    b.close()
    plan.close()
