"""The autotuner times the solves that its plans run: kernel timing, which takes the fused plane kernel apart, stays
off, and a chunk that takes the plane kernel away (its three separate kernels need twice the time on this grid) is not
picked."""
import pytest

import eddyproj
from eddyproj import autotune, grid

pytestmark = pytest.mark.gpu


def test_autotune_times_whole_solves(torch_cuda, monkeypatch):
    timed = []
    monkeypatch.setattr(eddyproj.Plan, "enable_timing", lambda self, on=True: timed.append(on))
    g = grid.make_grid(32, 24, 96, x_beta=1.4, z_beta=1.2)
    best, trace = autotune.autotune(g)
    assert not any(timed)
    ms = {t["value"]: t["ms"] for t in trace if t["param"] == "xsolve_chunk" and "ms" in t}
    print("autotune chunks", ms, best, flush=True)
    assert set(ms) == {4, 6, 8, 12, 16, 24, 32}
    # 32 rows to one lane: past the 16 that the plane kernel's line solves hold
    assert ms[32] > 1.3 * ms[12]
    assert best["xsolve_chunk"] != 32 and best["xsolve_chunk"] in ms
    assert best["fft_radix"] in (8, 4, 2)
