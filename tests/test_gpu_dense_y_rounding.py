"""Rounding of the dense inverse y transform, isolated: phi = S(x1, x2) (1 + 0.01 r(y)) on a period so long that the
solve divides every wavenumber of y alike, solved in FP32 without sweeps. The mean part of phi is 100 times the rest,
so a sum over the wavenumbers that takes it up first rounds at its size with every one of the L/2 terms that follow:
a noise along y of about sqrt(L/2) * 0.4 u, u = 2^-24 |S| (4.5 u at L = 254, 9 u at 1001). Taken up last, what is left
is a handful of roundings of 0.3 to 0.6 u each (the stored RHS, the last additions, the result) and the forward
transform's share of the wavenumbers above 20, 0.9 u at most: below 2 u together. The bound is 3 u. The (x1, x2) mean of each y
index, whose wavenumbers the long period leaves nearly singular, is taken out of the error."""
import numpy as np
import pytest

import eddyproj
from eddyproj import grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("l", [254, 509, 1001])
def test_inverse_sums_large_terms_last(torch_cuda, l):
    g = grid.make_grid(16, 16, l, lx3=1e5, x_stretch=False)
    rng = np.random.default_rng(l)
    x = (np.arange(16) + 0.5) / 16
    s = np.cos(np.pi * x)[:, None, None] * np.cos(np.pi * x)[None, None, :]
    r = rng.standard_normal(l)
    phi = np.zeros(g.shape(), order="F")
    phi[1:-1, 1:-1, 1:-1] = s * (1 + 0.01 * (r - r.mean()))[None, :, None]
    phi[:, 0], phi[:, -1] = phi[:, -2], phi[:, 1]
    plan = eddyproj.Plan(g)
    d = torch_cuda.zeros((g.nz, g.ny, g.nx), dtype=torch_cuda.float64, device="cuda")
    plan.laplacian(eddyproj.to_device(phi), d)
    plan.direct_refined(d, 0, residual=False)
    e = (eddyproj.to_host(d) - phi)[1:-1, 1:-1, 1:-1]
    plan.close()
    e = e - e.mean(axis=(0, 2), keepdims=True)
    f = np.fft.rfft(e, axis=1)
    f[:, :20] = 0
    e = np.fft.irfft(f, n=l, axis=1)
    rms = np.sqrt((e ** 2).mean(axis=1)) / (2.0 ** -24 * np.abs(s[:, 0]))
    rms = rms[np.abs(s[:, 0]) > 0.3]
    print("dense inverse", l, "%.2f u" % rms.mean(), flush=True)
    assert rms.mean() <= 3.0
