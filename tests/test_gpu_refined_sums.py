"""The sum of phi that closes the defect correction: every number of sweeps with and without the requested
residual (the closing pass and the fused last update), after another call has used the plan's reduction
slots, by radix FFT and by matrix products along y, and batches in both modes. The mean of phi is zero to
rounding and phi is the long-double oracle's within 20 times its FP32-contracted error (1e-4 a sweep, 1e-12
at the least); both closings agree to the same."""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gemm", [0, 1])
@pytest.mark.parametrize("sweeps", [0, 1, 2, 3])
def test_refined_mean(torch_cuda, sweeps, gemm):
    g = grid.make_grid(40, 24, 32, x_beta=1.3)
    u, v, w = configs.random_uniform_velocity(g, 7)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    tol = max(1e-12, 20 * 1e-4 ** (sweeps + 1))
    plan = eddyproj.Plan(g, tuning={"yfft_gemm": gemm})
    got = []
    for residual in (False, True):
        other = eddyproj.to_device(rhs * 3.0 + 1.0)  # leaves other sums behind
        plan.direct_refined(other, sweeps=1, residual=True)
        d = eddyproj.to_device(rhs)
        plan.direct_refined(d, sweeps=sweeps, residual=residual)
        torch_cuda.cuda.synchronize()
        phi = eddyproj.to_host(d)
        got.append(phi)
        err = rel_maxdiff_nomean(phi, ref)
        q = phi[1:-1, 1:-1, 1:-1]
        print("refined", sweeps, gemm, residual, "%.2e %.2e" % (err, abs(q.mean()) / np.abs(q).max()), flush=True)
        assert err <= tol
        assert abs(q.mean()) <= tol * np.abs(q).max()
    assert np.abs(got[0] - got[1]).max() <= tol * np.abs(got[1]).max()
    plan.close()
    if gemm:
        return
    for mode in (eddyproj.BATCH_BRANCHES, eddyproj.BATCH_QUEUES):
        b = eddyproj.Batch([g, g])
        b.set_mode(mode)
        ds = [eddyproj.to_device(rhs), eddyproj.to_device(-2.0 * rhs)]
        b.bind(ds)
        b.direct(eddyproj.EDDY_FP32_REFINE, sweeps)
        torch_cuda.cuda.synchronize()
        for d, f in zip(ds, (1.0, -2.0)):
            phi = eddyproj.to_host(d)
            q = phi[1:-1, 1:-1, 1:-1]
            assert rel_maxdiff_nomean(phi, f * ref) <= tol
            assert abs(q.mean()) <= tol * np.abs(q).max()
        b.close()
