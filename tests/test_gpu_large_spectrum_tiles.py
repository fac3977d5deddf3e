"""Spectra whose y transforms pass the caches by (the inverse from half the memory-side cache, the forward from all
of it): the projection of a plan against plans with narrower and wider y tiles in another order, and against the
one-launch batch, whose kernels read and write every spectrum through the caches; a solve of a stored RHS too.
Lengths of the radix FFT (the dense transform of others never passes the caches by): 258 and 143 MiB.

Tolerance: the same operations in the same order but for the sums of the solvability mean and the contraction of
differently inlined code: 1e-12 of the largest value, without the plain mean.
"""
import pytest

import eddyproj
from eddyproj import configs, grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(272, 256, 486), (272, 256, 270)])
def test_tiles_and_caches(torch_cuda, m, n, l):
    torch = torch_cuda
    g = grid.make_grid(m, n, l, x_beta=1.3)
    gen = torch.Generator(device="cuda").manual_seed(m - l)
    s = (g.nz, g.ny, g.nx)
    star = [torch.rand(s, dtype=torch.float64, device="cuda", generator=gen).sub_(0.5) for _ in range(3)]
    for a in star:  # periodic along y
        a[:, 0] = a[:, -2]
        a[:, -1] = a[:, 1]
    star[0][:, :, 0] = star[0][:, :, -2] = 0.0  # closed walls
    star[2][0] = star[2][-2] = 0.0

    def fresh():
        return [a.clone() for a in star], torch.zeros(s, dtype=torch.float64, device="cuda")

    def through(tuning):
        out, dp = fresh()
        plan = eddyproj.Plan(g, tuning=tuning)
        plan.project(*star, *out, dp, configs.DT)
        torch.cuda.synchronize()
        plan.close()
        return out, dp

    out, dp = through(None)
    plan = eddyproj.Plan(g)
    rhs = torch.zeros_like(dp)
    plan.divergence(*star, rhs, 1.0 / configs.DT)
    plan.direct(rhs)
    torch.cuda.synchronize()
    plan.close()
    others = [through({"yfft_pencils": 8, "yfft_iblock": 3}), through({"yfft_pencils": 32, "yfft_iblock": 2})]
    batch = eddyproj.Batch([g])
    batch.set_mode(eddyproj.BATCH_QUEUES)
    bo, bdp = fresh()
    batch.bind([bdp], *[[a] for a in star], *[[a] for a in bo])
    batch.project(configs.DT)
    torch.cuda.synchronize()
    batch.close()
    others += [(bo, bdp), (out, rhs)]
    c = (slice(1, -1),) * 3
    want = dp[c] - dp[c].mean()
    for o, d in others:
        got = d[c] - d[c].mean()
        err = float((got - want).abs().max() / want.abs().max())
        vel = max(float((x - y).abs().max()) for x, y in zip(o, out))
        print("large spectrum tiles", m, n, l, "%.1e %.1e" % (err, vel), flush=True)
        assert err <= 1e-12 and vel <= 1e-12
