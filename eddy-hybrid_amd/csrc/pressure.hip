// pressure.hip -- the pressure update that closes the substep after CORRECT
// (Eddy6.f:2772-2846):
//   P = P + DP, minus the implicit-viscous corrections when IMPLY / IMPLX are on
//     (:2777-2796, RU1 and the RVIMPLY / RVIMPLX masks per x1 index);
//   PREF = sum(P(IX1, JY1:JY2, KZ1)) / (NY-2) subtracted everywhere (:2801-2806);
//   ghost boundary values: x (:2813-2824, MP and the ITYPE(1) = 300 axis with JSYM), y
//   (:2829-2835, LP), z (:2843-2847, ITYPE(5) / ITYPE(6): 500 periodic, else Neumann).
//
// Two launches: the reference value (one workgroup), then the update. The reference applies its
// boundary copies one axis after the other over whole planes; every ghost value therefore equals +-P
// at one interior cell, found by mapping the z index, then the y index, then the x index (with its
// sign and the axis reflection). The thread of an interior cell writes the ghosts that copy it beside
// its own value, so that no pass over the shell waits for the interior to be done. Bound by memory at
// large sizes (512 x 256 x 256 0.163 -> 0.155 ms, 5.2 TB/s on its 24 B/cell; with the implicit y correction 0.201
// as before, 4.0 TB/s) and by its two dependent
// launches at small ones (203 x 101 x 90 0.0176 -> 0.0142 ms, 32 x 32 x 32 0.0120 -> 0.0078).
#include <algorithm>

#include "kernels.h"
#include "reduce_device.h"
#include "stencil_device.h"

namespace eddy {

// P + DP minus the implicit corrections at interior cell (I, J, K) (0-based with ghosts).
__device__ __forceinline__ double p_updated(const PressArgs& a, int I, int J, int K) {
    const Dims d = a.d;
    const size_t o = sidx(d, I, J, K);
    double v = a.p[o] + a.dp[o];
    if (a.imply) {
        const double r = a.dely * a.mt.rp[I];
        v = v - 0.5 * a.alfxdt * a.ru1 / (r * r) * (a.dp[o - d.nx] - 2. * a.dp[o] + a.dp[o + d.nx]) * a.rvy[I];
    }
    if (a.implx) {
        v = v - 0.5 * a.alfxdt * a.ru1 * a.mt.ap[I] / a.mt.rp[I] *
                    ((a.dp[o + 1] - a.dp[o]) * a.mt.au[I] * a.mt.ru[I] -
                     (a.dp[o] - a.dp[o - 1]) * a.mt.au[I - 1] * a.mt.ru[I - 1]) *
                    a.rvx[I];
    }
    return v;
}

// PREF = mean over the interior y rows of the updated P at (IX1, KZ1) -> red[RED_PREF].
__global__ void __launch_bounds__(256) k_pref(PressArgs a) {
    double s = 0.0;
    for (int J = 1 + threadIdx.x; J <= a.d.L; J += blockDim.x) s += p_updated(a, 1, J, 1);
    __shared__ double part[4];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < (int)(blockDim.x + 63) / 64; ++w) t += part[w];
        a.red[RED_PREF] = t / (double)a.d.L;
    }
}

// The value v of interior cell (I, J, K) and of every ghost that the boundary copies take from it:
// ghost planes 0 and n-1 of an axis copy interior planes lo and hi, composed z, y, x.
__device__ __forceinline__ void p_store(const PressArgs& a, int I, int J, int K, double v) {
    const Dims d = a.d;
    const int zlo = a.itype5 == 500 ? d.N : 1, zhi = a.itype6 == 500 ? 1 : d.N;
    const int ylo = a.lp == 0 ? d.L : 1, yhi = a.lp == 0 ? 1 : d.L;
    auto planes = [&](int i, int j, double x) {
        a.p[sidx(d, i, j, K)] = x;
        if (K == zlo) a.p[sidx(d, i, j, 0)] = x;
        if (K == zhi) a.p[sidx(d, i, j, d.nz - 1)] = x;
    };
    auto rows = [&](int i, int j, double x) {
        planes(i, j, x);
        if (j == ylo) planes(i, 0, x);
        if (j == yhi) planes(i, d.ny - 1, x);
    };
    rows(I, J, v);
    if (a.itype1 == 300) {  // axis: P(1,J,:) = P(IX1, JSYM(J), :), JSYM(J) = J + (NY-2)/2 mod the period
        if (I == 1) {
            const int j = J - d.L / 2;
            rows(0, j < 1 ? j + d.L : j, v);
        }
    } else if (a.mp == 0) {
        if (I == d.M) rows(0, J, v);
    } else if (I == 1) {
        rows(0, J, -v);
    }
    if (a.mp == 0) {
        if (I == 1) rows(d.nx - 1, J, v);
    } else if (I == d.M) {
        rows(d.nx - 1, J, -v);
    }
}

__global__ void __launch_bounds__(256) k_p_update(PressArgs a) {
    const int I = blockIdx.x * 64 + threadIdx.x + 1;
    const int J = blockIdx.y * 4 + threadIdx.y + 1;
    const int K = blockIdx.z + 1;
    if (I > a.d.M || J > a.d.L) return;
    p_store(a, I, J, K, p_updated(a, I, J, K) - a.red[RED_PREF]);
}

void launch_pressure_update(hipStream_t st, const PressArgs& a) {
    const Dims& d = a.d;
    hipLaunchKernelGGL(k_pref, dim3(1), dim3(256), 0, st, a);
    hipLaunchKernelGGL(k_p_update, dim3(ceil_div(d.M, 64), ceil_div(d.L, 4), d.N), dim3(64, 4, 1), 0, st, a);
}

}  // namespace eddy
