"""Transform lengths whose passes give a thread several butterflies (half-lengths with a factor 2, 3 or 4 beside larger
ones), along y and x2, whole and ragged tiles and batches, against the long-double oracle at the suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(70, 4, 36), (65, 4, 60), (33, 6, 72), (40, 4, 120), (20, 4, 150), (17, 4, 180),
                                   (33, 4, 216), (16, 4, 300), (18, 4, 360), (9, 4, 400), (70, 36, 4), (65, 60, 6),
                                   (40, 120, 4), (20, 180, 4), (33, 216, 4), (150, 300, 4), (17, 360, 4)])
def test_several_butterflies(torch_cuda, m, n, l):
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
        print("butterflies", m, n, l, "%.2e" % err, flush=True)
        assert err <= 1e-12
    plan.close()
    b = eddyproj.Batch([g])
    b.set_mode(eddyproj.BATCH_QUEUES)
    d = eddyproj.to_device(rhs)
    b.bind([d])
    b.direct()
    torch_cuda.cuda.synchronize()
    assert rel_maxdiff_nomean(eddyproj.to_host(d), ref) <= 1e-12
    b.close()
