"""The ghost shell that the pressure update's interior cells write: every boundary form of each axis (walls,
periodic, axis reflection over an even and an odd period, one-sided x2 copies) at the smallest and at ragged
sizes, against the oracle: interior within a rounding of PREF and of contracted multiply-adds (1e-14), each ghost the
oracle's copy of the same cells."""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid

pytestmark = pytest.mark.gpu

CASES = [(2, 4, 2, 1, 0, 0, 1, 1), (3, 4, 4, 0, 0, 0, 1, 1), (65, 4, 6, 1, 1, 0, 500, 500), (64, 5, 5, 0, 1, 0, 500, 1),
         (66, 6, 9, 1, 0, 0, 1, 500), (9, 4, 8, 1, 0, 300, 500, 500), (67, 4, 7, 1, 0, 300, 1, 1),
         (12, 4, 5, 0, 0, 300, 1, 500), (130, 7, 3, 0, 0, 0, 1, 1)]


@pytest.mark.parametrize("m,n,l,mp,lp,itype1,itype5,itype6", CASES)
def test_pressure_ghosts(torch_cuda, m, n, l, mp, lp, itype1, itype5, itype6):
    print("pressure ghosts", m, n, l, mp, lp, itype1, itype5, itype6, flush=True)
    g = grid.make_grid(m, n, l, x_beta=1.3, cyl=itype1 == 300, **({"lx3": 2 * np.pi} if itype1 == 300 else {}))
    g.mp, g.lp = mp, lp
    rng = np.random.default_rng(m + l)
    p = np.asfortranarray(rng.standard_normal(g.shape()))
    dp = np.asfortranarray(rng.standard_normal(g.shape()))
    uk = dict(itype1=itype1, itype5=itype5, itype6=itype6, implx=1, imply=1, ru1=0.01,
              rvimplx=np.ones(g.nx), rvimply=np.ones(g.nx))
    ref = oracle.pressure_update(g, p, dp, configs.DT, **uk)
    plan = eddyproj.Plan(g)
    plan.set_pressure_bc(**uk)
    dpd, pd = eddyproj.to_device(dp), eddyproj.to_device(p)
    plan.pressure_update(pd, dpd, configs.DT)
    torch_cuda.cuda.synchronize()
    got = eddyproj.to_host(pd)
    assert np.abs(got - ref).max() <= 1e-14 * np.abs(ref).max()
    plan.close()
