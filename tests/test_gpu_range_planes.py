"""The divergence range where a block takes one to eight planes and the last block fewer, rows of odd and even
length, Cartesian and cylindrical; against the extremes of the same divergence in plain torch.

Tolerance: three differences, four products, two quotients and two additions, each rounded at most at the size of
the terms' absolute values: 16 units in the last place of the largest sum of those.
"""
import pytest

import eddyproj
from eddyproj import grid

pytestmark = pytest.mark.gpu


# planes per block 1, 2, 3, 4, 7, 8 (the last blocks: 1, 1, 2, 1, 6, 1)
@pytest.mark.parametrize("cyl", [False, True])
@pytest.mark.parametrize("m,n,l", [(63, 5, 9), (255, 83, 200), (510, 131, 100), (254, 301, 120), (766, 97, 200),
                                   (401, 201, 212)])
def test_range(torch_cuda, m, n, l, cyl):
    torch = torch_cuda
    g = grid.make_grid(m, n, l, x_beta=1.3, cyl=cyl)
    gen = torch.Generator(device="cuda").manual_seed(m + n)
    u, v, w = (torch.rand((g.nz, g.ny, g.nx), dtype=torch.float64, device="cuda", generator=gen).sub_(0.5)
               for _ in range(3))
    plan = eddyproj.Plan(g)
    lo, hi = plan.div_minmax(u, v, w)
    plan.close()

    def dev(a, shape):
        return torch.as_tensor(a, device="cuda").view(shape)

    ap, bp, cp = dev(g.ap, (1, 1, -1)), dev(g.bp, (1, -1, 1)), dev(g.cp, (-1, 1, 1))
    rp, ru = dev(g.rp, (1, 1, -1)), dev(g.ru, (1, 1, -1))
    c = slice(1, -1)

    def total(sign, f):
        x = ap[:, :, c] * (f(ru * u)[c, c, 1:-1] + sign * f(ru * u)[c, c, :-2]) / rp[:, :, c]
        y = bp[:, c] * (f(v)[c, 1:-1, c] + sign * f(v)[c, :-2, c]) / rp[:, :, c]
        return x + y + cp[c] * (f(w)[1:-1, c, c] + sign * f(w)[:-2, c, c])

    d = total(-1.0, lambda a: a)
    tol = 16 * 2.0 ** -53 * float(total(1.0, torch.abs).abs().max())
    print("range", m, n, l, cyl, "%.3e %.3e tol %.1e" % (lo - float(d.min()), hi - float(d.max()), tol), flush=True)
    assert abs(lo - float(d.min())) <= tol and abs(hi - float(d.max())) <= tol
