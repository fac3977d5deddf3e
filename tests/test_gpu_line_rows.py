"""Line solves whose lanes hold 7 to 12 rows each, with and without padding at the line ends, 4, 2 and 1 lines
to a wave and a last wave that is not full, single and in a batch, against the long-double oracle at the
suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [97, 107, 121, 137, 144, 150, 176, 185, 193, 210, 250, 270, 288, 300, 333, 352, 370,
                               385, 440, 449, 513, 576, 600, 650, 704, 750])
def test_rows_per_lane(torch_cuda, m):
    g = grid.make_grid(m, 5, 6, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    plan = eddyproj.Plan(g)
    for timing in (False, True):  # the fused plane kernel where the plan takes it, and the separate ones
        plan.enable_timing(timing)
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        torch_cuda.cuda.synchronize()
        err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
        print("rows", m, "%.2e" % err, flush=True)
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
