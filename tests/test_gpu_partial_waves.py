"""Line solves whose last wave holds fewer lines than fit, after a solve that left NaN in every CU's LDS: lanes
without a line must not reach the others' results. 4 and 2 lines to a wave, 1 to 3 of them missing, splits with and
without padding and the general form; FP64, FP32 with sweeps and the one-launch batch, against the long-double oracle
at the suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def poison(torch_cuda):
    """A solve of an all-NaN RHS: its last kernel leaves 37 KB of NaN in the LDS of each of its workgroups, several
    to every CU."""
    g = grid.make_grid(256, 64, 256)
    plan = eddyproj.Plan(g)
    nan = torch_cuda.empty((g.nz, g.ny, g.nx), dtype=torch_cuda.float64, device="cuda")

    def run():
        plan.direct(nan.fill_(float("nan")))
    yield run
    plan.close()


# lines: 15 and 25 leave 3 and 1 of 4, 30 leaves 2; the small tiles of so few lines leave the poison in place
@pytest.mark.parametrize("n,l", [(3, 5), (5, 5), (5, 6)])
@pytest.mark.parametrize("m", [40, 101, 112, 128, 150, 185, 250, 333])
def test_missing_lines(torch_cuda, poison, m, n, l):
    g = grid.make_grid(m, n, l, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m + l)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)

    def check(what, solve):
        d = eddyproj.to_device(rhs)
        poison()
        solve(d)
        torch_cuda.cuda.synchronize()
        err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
        print("missing lines", m, n, l, what, "%.2e" % err, flush=True)
        assert err <= 1e-12  # also false for NaN

    plan = eddyproj.Plan(g)
    for timing in (False, True):  # the fused plane kernel where the plan takes it, and the separate ones
        plan.enable_timing(timing)
        check("fp64", plan.direct)
        check("fp32", lambda d: plan.direct_refined(d, 5, residual=False))
    plan.close()
    if l % 2 == 0:  # batches take even periodic lengths
        b = eddyproj.Batch([g])
        b.set_mode(eddyproj.BATCH_QUEUES)

        def batch(d):
            b.bind([d])
            b.direct()
        check("batch", batch)
        b.close()
