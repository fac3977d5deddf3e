"""The index maps of csrc/index_map.h, compiled for the host."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "eddy-hybrid_amd", "csrc")


def run(tmp_path, body, flags=()):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = str(tmp_path / "t.cpp"), str(tmp_path / "t")
    with open(src, "w") as f:
        f.write('#define __host__\n#define __device__\n#include "index_map.h"\n#include <cstdio>\n#include <vector>\n'
                "using namespace eddy;\n" + body)
    subprocess.run([cxx, "-std=c++17", "-O1", *flags, "-I", CSRC, src, "-o", exe], check=True)
    return subprocess.run([exe], capture_output=True, text=True, timeout=300)


def test_line_solve_order_keeps_each_xcds_eighth(tmp_path):
    """Every tile once, and each on the XCD (workgroup number modulo 8) that takes it in the forward order."""
    r = run(tmp_path, """
int main() {
    for (int n = 1; n < 3000; ++n) {
        std::vector<int> xcd(n), seen(n, 0);
        for (int b = 0; b < n; ++b) xcd[xcd_tile(b, n)] = b % 8;
        int last[8] = {n, n, n, n, n, n, n, n};
        for (int b = 0; b < n; ++b) {
            const int t = xcd_tile_back(b, n);
            if (t < 0 || t >= n || seen[t]++ || xcd[t] != b % 8 || t >= last[b % 8]) return printf("n %d b %d\\n", n, b), 1;
            last[b % 8] = t;
        }
    }
}
""")
    assert r.returncode == 0, r.stdout


def test_plane_pairs(tmp_path):
    """Every element number that CORRECT's and the divergence range's spans produce, and those that wrap below the
    plane's start (rows shorter than 16), against the division; without undefined arithmetic."""
    r = run(tmp_path, """
static bool check(int nx, int ny, unsigned r) {
    const int M = nx - 2, L = ny - 2;
    const Pair p = plane_pair(nx, M, L, r, row_reciprocal(nx));
    const unsigned i = r % (unsigned)nx, j = r / (unsigned)nx;
    const bool on = r < (unsigned)(nx * ny) && j >= 1 && j <= (unsigned)L && i <= (unsigned)M;
    if (p.on == on && (!on || (p.i == (int)i && p.j == (int)j))) return true;
    printf("nx %d ny %d r %u: %d %d %d\\n", nx, ny, r, p.i, p.j, (int)p.on);
    return false;
}
int main() {
    for (int nx = 4; nx < 1100; nx += nx < 80 ? 1 : 17)
        for (int ny = 4; ny < 40; ny += 5) {
            for (unsigned r = 0; r < (unsigned)(nx * ny) + 2048; ++r)
                if (!check(nx, ny, r)) return 1;
            for (unsigned below = 1; below <= 16; ++below)
                if (!check(nx, ny, 0u - below)) return 1;
        }
    for (unsigned r = 0; r < 1u << 29; r += 65521)  // the largest fields: rows and planes of 2^29 elements
        for (int nx : {4, 5, 66, 771, 2050, 130000})
            if (!check(nx, (1 << 29) / nx, r)) return 1;
}
""", ["-fsanitize=undefined", "-fno-sanitize-recover=all"])
    assert r.returncode == 0, r.stdout + r.stderr
