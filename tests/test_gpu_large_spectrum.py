"""Spectra beyond the memory-side cache (non-temporal stores and reads in the y transforms): the plan's solution
and projection against the same problem with a tile order and widths of their own, and the velocity's divergence
after CORRECT at rounding. 272 x 256 x 496 cells (276 MB), M a multiple of 16; 152 MB for the inverse alone."""
import pytest

import eddyproj
from eddyproj import configs, grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(272, 256, 496), (272, 256, 272)])
def test_large_spectrum(torch_cuda, m, n, l):
    torch = torch_cuda
    g = grid.make_grid(m, n, l, x_beta=1.3)
    gen = torch.Generator(device="cuda").manual_seed(m + l)
    s = (g.nz, g.ny, g.nx)
    star = [torch.rand(s, dtype=torch.float64, device="cuda", generator=gen).mul_(2).sub_(1) for _ in range(3)]
    for a in star:  # periodic along y
        a[:, 0] = a[:, -2]
        a[:, -1] = a[:, 1]
    star[0][:, :, 0] = star[0][:, :, -2] = 0.0  # closed walls
    star[2][0] = star[2][-2] = 0.0
    plan = eddyproj.Plan(g)
    lo, hi = plan.div_minmax(*star)
    scale = max(abs(lo), abs(hi))
    out = [a.clone() for a in star]
    dp = torch.zeros(s, dtype=torch.float64, device="cuda")
    plan.project(*star, *out, dp, configs.DT)
    lo, hi = plan.div_minmax(*out)
    print("large spectrum", m, n, l, "%.2e" % (max(abs(lo), abs(hi)) / scale), flush=True)
    assert max(abs(lo), abs(hi)) <= 1e-12 * scale
    # a stored RHS through the other forward form
    rhs = torch.zeros_like(dp)
    plan.divergence(*star, rhs, 1.0 / configs.DT)
    plan.direct(rhs)
    a, b = (x[1:-1, 1:-1, 1:-1] for x in (rhs, dp))
    a, b = a - a.mean(), b - b.mean()
    assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
    plan.close()
