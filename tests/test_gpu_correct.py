"""CORRECT over memory spans: rows of odd and even length, spans at and past whole blocks, every
face-range flag, fields that are not 16-byte aligned (the row kernel), and the projection's ghost
rows; against the oracle, entry by entry, the entries CORRECT leaves alone included.

Tolerance: u - g with both formed in FP64 in the oracle's operation order up to contraction: 4 ulp
of the largest value.
"""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid

pytestmark = pytest.mark.gpu

# (m, n, l, mp, lp, np): nx = 5, 64 (l*nx = one block of 1024 elements), 63, 514, 1026
CASES = [(3, 3, 4, 1, 0, 1), (62, 6, 16, 1, 0, 1), (61, 5, 17, 1, 0, 1), (61, 6, 34, 1, 1, 1), (512, 3, 9, 1, 0, 1),
         (1024, 4, 5, 1, 0, 1), (30, 8, 12, 0, 0, 1), (33, 7, 10, 1, 0, 0), (33, 6, 10, 0, 1, 0)]


def _shifted(torch, t, by):
    buf = torch.zeros(t.numel() + by, dtype=t.dtype, device=t.device)
    v = buf[by:].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("cyl", [False, True])
@pytest.mark.parametrize("m,n,l,mp,lp,np_", CASES)
def test_correct_spans(torch_cuda, m, n, l, mp, lp, np_, cyl):
    g = grid.make_grid(m, n, l, x_stretch=mp == 1, cyl=cyl and mp == 1)
    g.mp, g.lp, g.np = mp, lp, np_
    rng = np.random.default_rng(m + l)
    us, vs, ws, phi = (np.asfortranarray(rng.standard_normal(g.shape())) for _ in range(4))
    ref = oracle.correct(g, us, vs, ws, phi, 1e-3)
    plan = eddyproj.Plan(g)
    for by in (0, 1, 2):
        t = [_shifted(torch_cuda, eddyproj.to_device(a), by) for a in (us, vs, ws, phi)]
        out = [_shifted(torch_cuda, a, by) for a in t[:3]]
        plan.correct(*t[:3], *out, t[3], 1e-3)
        torch_cuda.cuda.synchronize()
        for a, b in zip(out, ref):
            np.testing.assert_allclose(eddyproj.to_host(a), b, rtol=0, atol=9e-16 * np.abs(b).max())
    plan.close()


@pytest.mark.parametrize("m,n,l", [(61, 5, 18), (62, 6, 16), (24, 4, 8)])
def test_projection_ghost_rows_and_alignment(torch_cuda, m, n, l):
    """The projection of aligned and unaligned fields, single and in a batch: the same fields."""
    g = grid.make_grid(m, n, l)
    vel = configs.random_uniform_velocity(g, 5)
    got = []
    for by in (0, 1):
        t = [_shifted(torch_cuda, eddyproj.to_device(a), by) for a in vel]
        o = [_shifted(torch_cuda, a, by) for a in t]
        dp = _shifted(torch_cuda, torch_cuda.zeros_like(t[0]), by)
        plan = eddyproj.Plan(g)
        plan.project(*t, *o, dp, configs.DT)
        torch_cuda.cuda.synchronize()
        got.append([eddyproj.to_host(a) for a in o])
        plan.close()
        for mode in (eddyproj.BATCH_BRANCHES, eddyproj.BATCH_QUEUES):
            bo = [_shifted(torch_cuda, a, by) for a in t]
            b = eddyproj.Batch([g])
            b.set_mode(mode)
            b.bind([dp], *[[a] for a in t], *[[a] for a in bo])
            b.project(configs.DT)
            torch_cuda.cuda.synchronize()
            got.append([eddyproj.to_host(a) for a in bo])
            b.close()
    for u, v, w in got:
        for a, b in zip((u, v, w), got[0]):
            np.testing.assert_allclose(a, b, rtol=0, atol=1e-12 * np.abs(b).max())
        # periodic images of the corrected faces
        np.testing.assert_array_equal(u[1:-2, 0, 1:-1], u[1:-2, -2, 1:-1])
        np.testing.assert_array_equal(v[1:-1, -1, 1:-1], v[1:-1, 1, 1:-1])
        np.testing.assert_array_equal(w[1:-1, -1, 1:-2], w[1:-1, 1, 1:-2])
