"""The resident loop's device arithmetic: the N(0,1) deviates against long double, and the divergence
range at the edges of its spans.

Deviates: a radius and a sine each within an ulp and one product: 3 ulp. Range: a handful of FP64
operations on values of the range's own size: 1e-14 of it.
"""
import numpy as np
import pytest

import eddyproj
import oracle
from eddyproj import configs, grid
from helpers import interior

pytestmark = pytest.mark.gpu


def _words(n, step, seed):
    m = np.uint64(0xffffffff)
    c = np.arange(n, dtype=np.uint64)
    x = [c & m, c >> np.uint64(32), np.full(n, step, np.uint64), np.zeros(n, np.uint64)]
    k0, k1 = seed, 0
    for _ in range(10):
        p0, p1 = x[0] * np.uint64(0xD2511F53), x[2] * np.uint64(0xCD9E8D57)
        x = [(p1 >> np.uint64(32)) ^ x[1] ^ np.uint64(k0), p1 & m, (p0 >> np.uint64(32)) ^ x[3] ^ np.uint64(k1), p0 & m]
        k0, k1 = (k0 + 0x9E3779B9) & 0xffffffff, (k1 + 0xBB67AE85) & 0xffffffff
    return x


@pytest.mark.parametrize("m,n,l,step", [(62, 62, 62, 0), (61, 30, 45, 12345), (253, 9, 66, 7)])
def test_deviates(torch_cuda, m, n, l, step):
    torch, ld = torch_cuda, np.longdouble
    g = grid.make_grid(m, n, l)
    plan = eddyproj.Plan(g)
    shape = (n + 2, l + 2, m + 2)
    zero = [torch.zeros(shape, dtype=torch.float64, device="cuda") for _ in range(3)]
    out = [torch.zeros_like(z) for z in zero]
    plan.perturb(*zero, *out, 1.0, 5, torch.tensor([step], dtype=torch.int32, device="cuda"))
    torch.cuda.synchronize()
    a = [(w.astype(ld) + ld(0.5)) / ld(2) ** 32 for w in _words(out[0].numel(), step, 5)]
    pi = ld("3.14159265358979323846264338327950288")
    y = [2 * t - 1 for t in (a[1], a[3])]  # the angle 2 pi t is pi (y + 1), y exact
    r0, r1 = np.sqrt(-2 * np.log(a[0])), np.sqrt(-2 * np.log(a[2]))
    h = [ld(0.5) - np.abs(t) for t in y]
    want = [-r0 * np.sin(pi * h[0]), -r0 * np.sign(y[0]) * np.sin(pi * (ld(0.5) - np.abs(h[0]))), -r1 * np.sin(pi * h[1])]
    at = np.arange(out[0].numel()).reshape(shape)[1:-2, 1:-1, 1:-2].ravel()
    for name, o, q in zip("uvw", out, want):
        got, q = o.cpu().numpy().ravel()[at].astype(ld), q[at]
        ulp = float((np.abs(got - q) / np.spacing(np.abs(q.astype(np.float64)))).max())
        print("deviates", m, n, l, step, name, "max %.2f ulp" % ulp, flush=True)
        assert ulp <= 3.0
    plan.close()


# (m, n, l): odd and even rows, spans at and past a block, more spans than x1 cells, groups of planes
# that do not fill
@pytest.mark.parametrize("cyl", [False, True])
@pytest.mark.parametrize("m,n,l", [(3, 3, 4), (62, 6, 16), (61, 5, 17), (3, 4, 1200), (510, 37, 30), (129, 67, 126)])
def test_divergence_range(torch_cuda, m, n, l, cyl):
    g = grid.make_grid(m, n, l, cyl=cyl)
    us, vs, ws = configs.random_uniform_velocity(g, m + n)
    d = interior(oracle.divergence(g, us, vs, ws))
    plan = eddyproj.Plan(g)
    for by in (0, 1):
        t = []
        for a in (us, vs, ws):
            x = eddyproj.to_device(a)
            buf = torch_cuda.zeros(x.numel() + by, dtype=x.dtype, device="cuda")
            buf[by:].copy_(x.view(-1))
            t.append(buf[by:].view(x.shape))
        lo, hi = plan.div_minmax(*t)
        tol = 1e-14 * max(abs(d.min()), abs(d.max()))
        assert abs(lo - d.min()) <= tol and abs(hi - d.max()) <= tol
    plan.close()
