"""The x1 line solve over its splits of a line into P lanes of Q rows: the exact splits with a kernel
of their own (Q = 6, 8, 10, 12, 16), the general ones, padded lines (P*Q > M), waves whose lines
span several y-modes (N below 64/P) and a last wave that is not full; FP64 against the long-double
oracle at the suite's 1e-12 or, for the longest lines, four times the FP64 oracle's own error (1.5e-12
at 1500 rows: the error grows with the row count), FP32 by its own residual.
"""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import interior, rel_maxdiff_nomean

pytestmark = pytest.mark.gpu

# (m, n, l, xsolve_chunk)
CASES = [(3, 4, 6, 12), (6, 6, 4, 12), (12, 4, 6, 12), (24, 14, 10, 6), (64, 10, 6, 8), (80, 6, 4, 10), (96, 6, 10, 12),
         (100, 10, 4, 12), (192, 6, 6, 12), (203, 6, 6, 12), (256, 10, 6, 16), (300, 4, 6, 12), (384, 6, 4, 12),
         (512, 4, 4, 8), (521, 4, 6, 12), (768, 4, 4, 12), (1024, 4, 4, 12), (1500, 4, 4, 12)]


@pytest.mark.parametrize("m,n,l,chunk", CASES)
def test_line_split(torch_cuda, m, n, l, chunk):
    g = grid.make_grid(m, n, l, x_beta=1.2)
    u, v, w = configs.random_uniform_velocity(g, m + n)
    rhs = configs.rhs_from_velocity(g, u, v, w)
    ref = oracle.direct(g, rhs, extended=True)
    tol = max(1e-12, 4 * rel_maxdiff_nomean(oracle.direct(g, rhs), ref))
    plan = eddyproj.Plan(g, tuning={"xsolve_chunk": chunk})
    d = eddyproj.to_device(rhs)
    plan.direct(d)
    torch_cuda.cuda.synchronize()
    err = rel_maxdiff_nomean(eddyproj.to_host(d), ref)
    print("line split", m, n, l, chunk, "%.2e" % err, flush=True)
    assert err <= tol
    d = eddyproj.to_device(rhs)
    plan.direct_refined(d, sweeps=3)
    phi = eddyproj.to_host(d)
    b = interior(rhs)
    res = float(np.linalg.norm(b - interior(oracle.laplacian(g, phi))) / np.linalg.norm(b))
    print("  fp32 + 3 sweeps residual %.2e" % res, flush=True)
    assert res <= 1e-10
    plan.close()


def test_batch_line_classes(torch_cuda):
    """One batch that holds every exact class and general ones: more classes than four."""
    sizes = [(24, 6, 8), (64, 10, 8), (80, 6, 8), (96, 6, 10), (100, 10, 4), (256, 6, 6), (6, 6, 4), (521, 4, 6)]
    tun = [{"xsolve_chunk": c} for c in (6, 8, 10, 12, 12, 16, 12, 32)]
    for mode in (eddyproj.BATCH_BRANCHES, eddyproj.BATCH_QUEUES):
        grids = [grid.make_grid(*s, x_beta=1.2) for s in sizes]
        rhs = [configs.rhs_from_velocity(g, *configs.random_uniform_velocity(g, 7 + i)) for i, g in enumerate(grids)]
        b = eddyproj.Batch(grids, tuning=tun)
        b.set_mode(mode)
        dps = [eddyproj.to_device(r) for r in rhs]
        b.bind(dps)
        b.direct()
        torch_cuda.cuda.synchronize()
        for g, r, dp in zip(grids, rhs, dps):
            err = rel_maxdiff_nomean(eddyproj.to_host(dp), oracle.direct(g, r, extended=True))
            assert err <= 1e-12, (mode, g.M, err)
        b.close()
