"""CORRECT of fields just inside and just past the sizes at which its velocities are read past the caches (7 fields of
64 MiB together) and its blocks are dealt in runs (256 MiB), single and as a batch of one, against the oracle at 4 ulp
of the largest value."""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,l", [(100, 100, 108), (104, 104, 108), (160, 160, 180), (164, 160, 180)])
def test_correct_at_the_cache_size(torch_cuda, m, n, l):
    g = grid.make_grid(m, n, l)
    rng = np.random.default_rng(m)
    us, vs, ws, phi = (np.asfortranarray(rng.standard_normal(g.shape())) for _ in range(4))
    t = [eddyproj.to_device(a) for a in (us, vs, ws)]
    out = [a.clone() for a in t]
    plan = eddyproj.Plan(g)
    plan.correct(*t, *out, eddyproj.to_device(phi), 1e-3)
    torch_cuda.cuda.synchronize()
    for a, b in zip(out, oracle.correct(g, us, vs, ws, phi, 1e-3)):
        np.testing.assert_allclose(eddyproj.to_host(a), b, rtol=0, atol=9e-16 * np.abs(b).max())
    # the same kernels from a batch's jobs
    dps, outs = [], []
    for mode in (eddyproj.BATCH_BRANCHES, eddyproj.BATCH_QUEUES):
        dps.append(torch_cuda.zeros_like(t[0]))
        outs.append([a.clone() for a in t])
        b = eddyproj.Batch([g])
        b.set_mode(mode)
        b.bind([dps[-1]], *[[a] for a in t], *[[a] for a in outs[-1]])
        b.project(configs.DT)
        torch_cuda.cuda.synchronize()
        b.close()
    plan.close()
    for a, b in zip(*outs):
        assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
