// zplane.hip -- one y-mode's whole plane in one workgroup: the x2 transform, the x1 line solves
// and the inverse x2 transform (ztrans.hip, xsolve.hip) with the plane in LDS between them, for
// planes that fit (M * N up to about 17,000 FP64 values).
//
// The plane is read once and written once where the three kernels make six passes over it, and two
// launches go. Inside, the waves own lines: the cosine transform's FFT passes and packing steps run
// on a wave's own pencils without workgroup barriers, the line solve on its own lines, so that five
// barriers separate the phases of a plane (load, transform, solve, inverse, store).
//
// Cosine transform (uniform x2): TI = M complex rows of length N/2 as in ztrans.hip, transformed in
// place; the packing step leaves X_m at the real part of slot m (m < N/2), X_{N/2} at the
// imaginary part of slot 0 and X_m at the imaginary part of slot N - m (m > N/2), which its inverse
// reads back.
// Dense transform (stretched or odd x2, M and N below 128): Y = F X and X = Q Y as matrix-core
// products, X straight from and to memory, Y (rows m, x1 contiguous) in LDS.
#include <algorithm>

#include "fft_device.h"
#include "kernels.h"
#include "mma_device.h"
#include "reduce_device.h"
#include "stencil_device.h"
#include "xsolve_device.h"

namespace eddy {

template <typename T>
struct PlaneArgs {
    T* S;
    MeanShift shift;  // the zero y-mode loses L times this mean
    FftPlan fp;       // complex FFT of length N/2 (cosine transform)
    XArgs<T> x;       // dims, tables and the partition of the lines
    int ld;           // LDS row pitch
    int pw;           // pencils per wave of an FFT call
    int j0;           // first y-mode of this launch
    unsigned rM;      // ceil(2^32 / M)
};

constexpr int kPlaneThreads = 1024;
constexpr int kPlaneSmall = 6144;  // planes up to this take 512 threads, two to a CU
constexpr size_t kPlaneLds = 160 * 1024 - 512;  // beside the static reduction scratch

// The lane index as a value the compiler cannot see through: inside the loops over a wave's pencils
// and lines it keeps every lane-dependent address of the loop body (several FFT plans, their
// twiddles) from being computed ahead of the loop and held in registers across it (66 to 228
// spilled registers at the 128 of a 1024-thread workgroup).
__device__ __forceinline__ int opaque(int lane) {
    asm volatile("" : "+v"(lane));
    return lane;
}

// The line solves of the plane; at(m, i) is the LDS element of x2 mode m and x1 row i. The line
// sums go to lsum when it is not null.
template <typename T, int QMAX, int ROWS, typename At>
__device__ __forceinline__ void plane_solve(const XArgs<T>& x, int j, T* lsum, At at) {
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int P = x.P, Q = ROWS != XR_ANY ? QMAX : x.Q, LW = 64 / P, N = x.d.N;
    const T akj = x.tb.akj[j];
    for (int b = __builtin_amdgcn_readfirstlane(w); b * LW < N; b += nw) {
        const int lane = opaque(threadIdx.x & 63);
        const int lw = lane / P, p = lane - lw * P;
        const int m = min(b * LW + lw, N - 1);
        const bool own = b * LW + lw < N;
        const T lam = x.tb.lam[m];
        T part = xsolve_lines<T, QMAX, ROWS, false>(
            x, p, lane, akj, lam, j == 0 && m == x.d.null_m,
            [&](int r) { return at(m, ROWS == XR_EXACT ? p * Q + r : min(p * Q + r, x.d.M - 1)); },
            [&](int r, T v) {
                if (own && (ROWS == XR_EXACT || p * Q + r < x.d.M)) at(m, p * Q + r) = v;
            });
        if (lsum) {
            for (int off = P >> 1; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
            if (own && p == 0) lsum[m] = part;
        }
    }
}

// Plain-mean correction of the zero y-mode (direct.f:894-898), as mean_delta in ztrans.hip, from
// the plane's own line sums; every thread calls it.
template <typename T>
__device__ __forceinline__ T plane_delta(const XArgs<T>& x, const T* lsum, double* scratch) {
    double s = 0.0;
    for (int m = threadIdx.x; m < x.d.N; m += blockDim.x) s += (double)x.tb.wsum[m] * (double)lsum[m];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) scratch[threadIdx.x >> 6] = s;
    __syncthreads();
    double tot = 0.0;
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) tot += scratch[w];
    return T(-tot / ((double)x.tb.wsum[x.d.null_m] * (double)x.d.M));
}

template <typename T, int QMAX, int ROWS>
__global__ void __launch_bounds__(kPlaneThreads) k_zplane_dct(PlaneArgs<T> a) {
    extern __shared__ __align__(16) unsigned char plane_lds[];
    __shared__ double scratch[16];
    const Dims d = a.x.d;
    const int M = d.M, N = d.N, H = N / 2, ld = a.ld;
    const int tid = threadIdx.x, nthr = blockDim.x, lane0 = tid & 63, nw = nthr >> 6;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = a.j0 + blockIdx.x;
    T* const Ar = reinterpret_cast<T*>(plane_lds);
    T* const Ai = Ar + M * ld;
    T* const twc_r = Ai + M * ld;  // H
    T* const twc_i = twc_r + H;
    T* const twr_r = twc_i + H;    // H + 1
    T* const twr_i = twr_r + H + 1;
    T* const dct_r = twr_i + H + 1;  // N
    T* const dct_i = dct_r + N;
    T* const lsum = dct_i + N;       // N
    T* const plane = a.S + (size_t)M * (size_t)N * (size_t)j;
    const Tables<T>& tb = a.x.tb;
    for (int t = tid; t < N; t += nthr) {
        if (t < H) {
            twc_r[t] = tb.ztwc_re[t];
            twc_i[t] = tb.ztwc_im[t];
        }
        dct_r[t] = tb.zdct_re[t];
        dct_i[t] = tb.zdct_im[t];
    }
    for (int t = tid; t <= H; t += nthr) {
        twr_r[t] = tb.ztwr_re[t];
        twr_i[t] = tb.ztwr_im[t];
    }
    const T zshift = j == 0 ? T((double)d.L * mean_shift(a.shift, scratch)) : T(0);

    // The plane is contiguous in S; row k goes to Makhoul position p(k) (ztrans.hip)
    const int MN = M * N;
    constexpr int U = 8;
    for (int e0 = tid; e0 < MN; e0 += nthr * U) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = ld_off(plane, (unsigned)sizeof(T) * (unsigned)min(e0 + u * nthr, MN - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int e = e0 + u * nthr;
            if (e >= MN) continue;
            const int k = (int)__umulhi((unsigned)e, a.rM), i = e - k * M;
            const int p = (k & 1) ? N - 1 - (k >> 1) : k >> 1;
            ((p & 1) ? Ai : Ar)[i * ld + pidx(p >> 1)] = v[u] - zshift;
        }
    }
    __syncthreads();

    // the wave's pencils: FFT, then the packing in place (pencil, q <= H/2)
    const int half = H / 2, lp = 64 / a.pw;  // lanes per pencil in the packing steps
    for (int i0 = w * a.pw; i0 < M; i0 += nw * a.pw) {
        const int np = min(a.pw, M - i0), lane = opaque(lane0);
        if (H > 1) cfft_lds<T, true>(Ar + i0 * ld, Ai + i0 * ld, ld, np, a.fp, twc_r, twc_i, T(-1), lane, 64);
        const int ii = lane / lp;
        for (int q = ii < np ? lane - ii * lp : half + 1; q <= half; q += lp) {
            T* const zr = Ar + (i0 + ii) * ld;
            T* const zi = Ai + (i0 + ii) * ld;
            const int qb = H - q, kb = q == 0 ? 0 : qb;
            const T zar = zr[pidx(q)], zai = zi[pidx(q)], zbr = zr[pidx(kb)], zbi = zi[pidx(kb)];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int m = s ? qb : q;
                if (s && qb == q) break;
                const T pr = s ? zbr : zar, pi = s ? zbi : zai;
                const T cr = s ? zar : zbr, ci = s ? -zai : -zbi;
                const T er = T(0.5) * (pr + cr), ei = T(0.5) * (pi + ci);
                const T dr = T(0.5) * (pr - cr), di = T(0.5) * (pi - ci);
                const T wr = twr_r[m], wi = twr_i[m];
                const T vr = er + wr * di + wi * dr, vi = ei - (wr * dr - wi * di);
                const T x = dct_r[m] * vr - dct_i[m] * vi;
                if (m == H) zi[0] = x;
                else zr[pidx(m)] = x;
                if (m > 0 && m < H) zi[pidx(m)] = dct_r[N - m] * vr + dct_i[N - m] * vi;
            }
        }
        fft_sync<true>();
    }
    __syncthreads();

    plane_solve<T, QMAX, ROWS>(a.x, j, j == 0 ? lsum : nullptr, [&](int m, int i) -> T& {
        return m < H ? Ar[i * ld + pidx(m)] : Ai[i * ld + (m == H ? 0 : pidx(N - m))];
    });
    __syncthreads();
    T delta = T(0);
    if (j == 0) {
        delta = plane_delta(a.x, lsum, scratch);
        __syncthreads();
    }

    // V and Z' of the wave's pencils in place, inverse FFT (zdct_inv_tile's arithmetic)
    const T invN = T(1) / T(N);
    const int nm = j == 0 ? d.null_m : -1;
    for (int i0 = w * a.pw; i0 < M; i0 += nw * a.pw) {
        const int np = min(a.pw, M - i0), lane = opaque(lane0);
        const int ii = lane / lp;
        for (int q = ii < np ? lane - ii * lp : half + 1; q <= half; q += lp) {
            T* const zr = Ar + (i0 + ii) * ld;
            T* const zi = Ai + (i0 + ii) * ld;
            const int qb = H - q;
            // X_q, X_{N-q} (X_N = 0), X_{H-q}, X_{H+q}
            T x[4];
            x[0] = zr[pidx(q)];
            x[1] = q ? zi[pidx(q)] : T(0);
            x[2] = q ? zr[pidx(qb)] : zi[0];
            x[3] = q ? zi[pidx(qb)] : x[2];
            const int ms[4] = {q, N - q, qb, H + q};
#pragma unroll
            for (int c = 0; c < 4; ++c) x[c] += ms[c] == nm ? delta : T(0);
            T vr[2], vi[2];
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int m = s ? qb : q;
                const T xr = x[2 * s], xi = -x[2 * s + 1];
                const T cr = dct_r[m], ci = -dct_i[m];
                vr[s] = cr * xr - ci * xi;
                vi[s] = (m == 0 || m == H) ? T(0) : cr * xi + ci * xr;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int kk = s ? qb : q;
                if (kk >= H || (s && qb == q)) continue;
                const T xr = vr[s], xi = vi[s];
                const T yr = vr[1 - s], yi = -vi[1 - s];
                const T sr = xr + yr, si = xi + yi;
                const T dr = xr - yr, di = xi - yi;
                const T wr = twr_r[kk], wi = -twr_i[kk];
                zr[pidx(kk)] = (sr - (wr * di + wi * dr)) * invN;
                zi[pidx(kk)] = (si + (wr * dr - wi * di)) * invN;
            }
        }
        fft_sync<true>();
        if (H > 1) cfft_lds<T, true>(Ar + i0 * ld, Ai + i0 * ld, ld, np, a.fp, twc_r, twc_i, T(1), lane, 64);
    }
    __syncthreads();
    for (int e = tid; e < MN; e += nthr) {
        const int k = (int)__umulhi((unsigned)e, a.rM), i = e - k * M;
        const int p = (k & 1) ? N - 1 - (k >> 1) : k >> 1;
        st_off(plane, (unsigned)sizeof(T) * (unsigned)e, ((p & 1) ? Ai : Ar)[i * ld + pidx(p >> 1)]);
    }
}

// out(o, i) = sum_s A(s, o) in(s, i) for 16 outputs o of block rb (`NB` consecutive blocks) and 16
// lines: A row-major s * N + o in memory, in(s) the operand of contraction index s for this lane.
template <typename T, int NB, typename In>
__device__ __forceinline__ void dense_block(const T* __restrict__ A, int N, int rb, int lane, In in,
                                            typename Mma<T>::v4 (&acc)[NB]) {
    const int x = lane & 15, q = lane >> 4;
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = typename Mma<T>::v4{T(0), T(0), T(0), T(0)};
    constexpr int U = 4;  // steps loaded ahead
    for (int s0 = 0; s0 < N; s0 += 4 * U) {
        T m[U][NB], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(s0 + 4 * u + q, N - 1);
            v[u] = in(s);
#pragma unroll
            for (int b = 0; b < NB; ++b) m[u][b] = A[(size_t)s * N + min(16 * (rb + b) + x, N - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // outputs past N are never used; contraction indices past N enter as 0 * in(N - 1)
            const bool ok = s0 + 4 * u + q < N;
            if (s0 + 4 * u < N)
#pragma unroll
                for (int b = 0; b < NB; ++b) acc[b] = Mma<T>::run(ok ? m[u][b] : T(0), ok ? v[u] : T(0), acc[b]);
        }
    }
}

template <typename T, int QMAX, int ROWS>
__global__ void __launch_bounds__(kPlaneThreads) k_zplane_dense(PlaneArgs<T> a) {
    extern __shared__ __align__(16) unsigned char plane_lds[];
    __shared__ double scratch[16];
    const Dims d = a.x.d;
    const int M = d.M, N = d.N, ld = a.ld;
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int j = a.j0 + blockIdx.x;
    T* const Y = reinterpret_cast<T*>(plane_lds);  // N rows of pitch ld
    T* const lsum = Y + N * ld;
    T* const plane = a.S + (size_t)M * (size_t)N * (size_t)j;
    const T zshift = j == 0 ? T((double)d.L * mean_shift(a.shift, scratch)) : T(0);
    constexpr int NB = 2;
    typedef typename Mma<T>::v4 v4;
    // item: 16 lines by NB blocks of 16 outputs
    const int ncb = (M + 15) >> 4, nrb = ((N + 15) >> 4), nrg = (nrb + NB - 1) / NB;
    const int x = lane & 15, q = lane >> 4;
    for (int it = w; it < ncb * nrg; it += nw) {
        const int rb = NB * (it / ncb), i = 16 * (it % ncb) + x;
        const T* col = plane + min(i, M - 1);
        v4 acc[NB];
        dense_block<T, NB>(a.x.tb.qf, N, rb, lane, [&](int s) { return col[s * M] - zshift; }, acc);
        if (i < M)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int m = 16 * (rb + b) + Mma<T>::row(q, v);
                    if (m < N) Y[m * ld + i] = acc[b][v];
                }
    }
    __syncthreads();
    plane_solve<T, QMAX, ROWS>(a.x, j, j == 0 ? lsum : nullptr, [&](int m, int i) -> T& { return Y[m * ld + i]; });
    __syncthreads();
    T delta = T(0);
    if (j == 0) delta = plane_delta(a.x, lsum, scratch);
    const int nm = j == 0 ? d.null_m : -1;
    for (int it = w; it < ncb * nrg; it += nw) {
        const int rb = NB * (it / ncb), i = 16 * (it % ncb) + x;
        const T* col = Y + min(i, M - 1);
        v4 acc[NB];
        dense_block<T, NB>(a.x.tb.qiT, N, rb, lane, [&](int s) { return col[s * ld] + (s == nm ? delta : T(0)); }, acc);
        if (i < M)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int k = 16 * (rb + b) + Mma<T>::row(q, v);
                    if (k < N) plane[k * M + i] = acc[b][v];
                }
    }
}

// LDS row pitch: the cosine rows odd (lanes of one x2 slot and consecutive x1), the dense rows
// 16 mod 32 (the two contraction indices of a half-wave's operand read in distinct banks).
static int plane_ld(const Dims& d, int dense) {
    if (!dense) return fft_ld(d.N / 2) | 1;
    const int l = ((d.M + 15) / 16) * 16;
    return l % 32 ? l : l + 16;
}

static size_t plane_lds_bytes(const Dims& d, int dense, size_t tsz) {
    const size_t ld = plane_ld(d, dense);
    return (dense ? (size_t)d.N * ld + d.N : 2 * (size_t)d.M * ld + 5 * (size_t)d.N + 2) * tsz;
}

// When the planes go through one workgroup each. The dense transform always gains where it fits
// (solves, three kernels against one: 32 x 24 x 96 0.034 -> 0.019 ms, 100 x 60 x 128 0.088 -> 0.044, 127 x 127 x 16 0.087 ->
// 0.080: its products move from the vector ALUs to the matrix cores too). The cosine form's work is bound by the
// issue of the one CU a plane runs on, so it pays where launches and latency rule or where the planes fill the CUs.
// Solves with the three kernels and with the one, ratio of the times:
//   planes up to 3072, any L: 48 x 48 0.85 to 0.95, 30 x 90 0.87 to 0.96, 96 x 32 0.90 to 0.97, 48 x 64 0.91 to 0.99; past it
//   64 x 64 x 32 1.09, 32 x 128 x 16 1.03;
//   larger ones from the L where they break even, 48 + plane / 86 (a line through 64 x 64 x 80 1.02, x 96 0.99,
//   x 144 0.90; 96 x 64 x 112 1.02, x 144 0.90; 64 x 128 x 112 1.05, x 144 0.91; 128 x 96 x 176 1.00, x 208 0.94;
//   128 x 128 x 192 1.01, x 240 0.90; 120 x 120 x 192 1.05, x 240 0.93);
//   planes past 6144 run on 1024 threads, one to a CU, and a second round of them loses: L = 288 1.07 to 1.23
//   (96 x 64 x 640, two to a CU, 0.94);
//   run-time FFT passes that hold a radix of 2 lose: 100 x 60 (N/2 = 30) x 128 1.17, x 208 1.00; 160 x 100 x 256 1.11.
// The FP32 sweeps follow the FP64 rule and its LDS (0.87 to 1.05 on the taken side).
bool zplane_fits(const Dims& d, const FftPlan& fpz, int dense, int chunk) {
    int P = 0, Q = 0;
    if (d.cyc_x || !xsolve_partition(d.M, chunk, P, Q) || Q > 16) return false;
    if (plane_lds_bytes(d, dense, sizeof(double)) > kPlaneLds) return false;
    if (dense) return d.M < 128 && d.N < 128;
    // a wave's FFT call holds whole pencils, one butterfly per lane and pass
    if (fpz.n / min_radix(fpz) > 64) return false;
    const int plane = d.M * d.N;
    if (plane <= 3072) return true;
    if (min_radix(fpz) < 3 && fpz.n > 8) return false;
    return plane <= 86 * (d.L - 48) && (plane <= kPlaneSmall || d.L <= 256);
}

template <typename T>
void launch_zplane(hipStream_t st, const Dims& d, const FftPlan& fpz, const Tables<T>& tb, T* S, int dense, int chunk,
                   const MeanShift& shift, int j0, int nj) {
    PlaneArgs<T> a{};
    a.S = S;
    a.shift = shift;
    a.fp = fpz;
    a.x.d = d;
    a.x.tb = tb;
    xsolve_partition(d.M, chunk, a.x.P, a.x.Q);
    a.ld = plane_ld(d, dense);
    a.j0 = j0;
    a.rM = (unsigned)(((1ull << 32) + d.M - 1) / d.M);
    const size_t lds = plane_lds_bytes(d, dense, sizeof(T));
    // 512 threads for the small planes (64 x 64 x 32: 0.0353 ms, 0.0360 with 1024)
    const int nthr = d.M * d.N <= kPlaneSmall ? 512 : kPlaneThreads;
    a.pw = dense ? 1 : std::max(1, 64 / std::max(1, fpz.n / min_radix(fpz)));
    xsolve_dispatch(xsolve_class(d.M, a.x.P, a.x.Q, false), [&](auto qmax, auto rows) {
        constexpr int QMAX = decltype(qmax)::value;
        if constexpr (QMAX <= 16) {
            auto go = [&](auto fn) {
                (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
                hipLaunchKernelGGL(fn, dim3(nj), dim3(nthr), lds, st, a);
            };
            if (dense) go(k_zplane_dense<T, QMAX, decltype(rows)::value>);
            else go(k_zplane_dct<T, QMAX, decltype(rows)::value>);
        }
    });
}

template void launch_zplane<double>(hipStream_t, const Dims&, const FftPlan&, const Tables<double>&, double*, int, int,
                                    const MeanShift&, int, int);
template void launch_zplane<float>(hipStream_t, const Dims&, const FftPlan&, const Tables<float>&, float*, int, int,
                                   const MeanShift&, int, int);

}  // namespace eddy
