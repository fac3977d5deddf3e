"""The plan's own transform tiles on both sides of its workgroup counts, where tiles are ragged and where they are
not, by radix FFT and dense y transforms: the same problem with every requested width and with the plan's, against the
long-double oracle at the suite's 1e-12."""
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import rel_maxdiff_nomean

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(17, 40, 16), (47, 54, 16), (64, 40, 16), (33, 80, 12), (70, 80, 8), (64, 160, 16),
                                   (33, 80, 14), (90, 160, 11), (40, 12, 130)])
def test_tile_widths(torch_cuda, m, n, l):
    g = grid.make_grid(m, n, l, x_beta=1.4)
    u, v, w = configs.random_uniform_velocity(g, m + n + l)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    for width in (0, 16, 32, 64):
        plan = eddyproj.Plan(g, tuning=dict(yfft_pencils=width, ztrans_pencils=width))
        plan.enable_timing(True)  # the x2 transforms as kernels of their own
        d = eddyproj.to_device(rhs)
        plan.direct(d)
        torch_cuda.cuda.synchronize()
        err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
        print("tile widths", m, n, l, width, "%.2e" % err, flush=True)
        assert err <= 1e-12
        plan.close()
