// fft_device.h -- batched complex FFTs in LDS (Stockham autosort, radix 2/3/4/5/8) and the
// real-FFT packing used by the y-transform (fftpack convention, src/fftpack.f:140-240) and
// the x2 DCT.
//
// A workgroup holds `P` independent length-n complex sequences in ONE LDS buffer (split re/im
// arrays, row stride `ld`) and transforms them in place: each radix pass loads every
// butterfly into registers, synchronises, then stores. Twiddles come from a table
// tw[t] = exp(-2 pi i t / n), t < n (conjugated for the inverse).
#pragma once

#include <algorithm>
#include <initializer_list>

#include "common.h"

namespace eddy {

// LDS rows of the FFT buffers are padded by one element per 8 (index x -> x + x/8): the
// Stockham writes stride by the radix and by 8*R, which would otherwise land many lanes of a
// wave on one LDS bank. A row holding indices 0..n needs fft_ld(n) elements.
__device__ __forceinline__ int pidx(int x) { return x + (x >> 3); }
__host__ __device__ inline int fft_ld(int n) { return n + (n >> 3) + 2; }

template <typename T>
struct Cx {
    T re, im;
};

template <typename T>
__device__ __forceinline__ Cx<T> cmul(Cx<T> a, Cx<T> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

// multiply by dir*i  (dir = -1 forward, +1 inverse)
template <typename T>
__device__ __forceinline__ Cx<T> mul_di(Cx<T> a, T dir) {
    return {-dir * a.im, dir * a.re};
}

template <typename T>
__device__ __forceinline__ void dft2(Cx<T>* v) {
    Cx<T> a = v[0], b = v[1];
    v[0] = {a.re + b.re, a.im + b.im};
    v[1] = {a.re - b.re, a.im - b.im};
}

template <typename T>
__device__ __forceinline__ void dft4(Cx<T>* v, T dir) {
    Cx<T> s02 = {v[0].re + v[2].re, v[0].im + v[2].im};
    Cx<T> d02 = {v[0].re - v[2].re, v[0].im - v[2].im};
    Cx<T> s13 = {v[1].re + v[3].re, v[1].im + v[3].im};
    Cx<T> d13 = mul_di(Cx<T>{v[1].re - v[3].re, v[1].im - v[3].im}, dir);
    v[0] = {s02.re + s13.re, s02.im + s13.im};
    v[2] = {s02.re - s13.re, s02.im - s13.im};
    v[1] = {d02.re + d13.re, d02.im + d13.im};
    v[3] = {d02.re - d13.re, d02.im - d13.im};
}

template <typename T>
__device__ __forceinline__ void dft3(Cx<T>* v, T dir) {
    const T h = T(0.86602540378443864676);  // sin(2 pi/3)
    Cx<T> t = {v[1].re + v[2].re, v[1].im + v[2].im};
    Cx<T> u = {v[1].re - v[2].re, v[1].im - v[2].im};
    Cx<T> a = {v[0].re - T(0.5) * t.re, v[0].im - T(0.5) * t.im};
    Cx<T> b = mul_di(Cx<T>{h * u.re, h * u.im}, dir);
    v[0] = {v[0].re + t.re, v[0].im + t.im};
    v[1] = {a.re + b.re, a.im + b.im};
    v[2] = {a.re - b.re, a.im - b.im};
}

template <typename T>
__device__ __forceinline__ void dft5(Cx<T>* v, T dir) {
    const T c1 = T(0.30901699437494742410);   // cos(2 pi/5)
    const T c2 = T(-0.80901699437494742410);  // cos(4 pi/5)
    const T s1 = T(0.95105651629515357212);   // sin(2 pi/5)
    const T s2 = T(0.58778525229247312917);   // sin(4 pi/5)
    Cx<T> t1 = {v[1].re + v[4].re, v[1].im + v[4].im};
    Cx<T> t2 = {v[2].re + v[3].re, v[2].im + v[3].im};
    Cx<T> u1 = {v[1].re - v[4].re, v[1].im - v[4].im};
    Cx<T> u2 = {v[2].re - v[3].re, v[2].im - v[3].im};
    Cx<T> a1 = {v[0].re + c1 * t1.re + c2 * t2.re, v[0].im + c1 * t1.im + c2 * t2.im};
    Cx<T> a2 = {v[0].re + c2 * t1.re + c1 * t2.re, v[0].im + c2 * t1.im + c1 * t2.im};
    Cx<T> b1 = mul_di(Cx<T>{s1 * u1.re + s2 * u2.re, s1 * u1.im + s2 * u2.im}, dir);
    Cx<T> b2 = mul_di(Cx<T>{s2 * u1.re - s1 * u2.re, s2 * u1.im - s1 * u2.im}, dir);
    v[0] = {v[0].re + t1.re + t2.re, v[0].im + t1.im + t2.im};
    v[1] = {a1.re + b1.re, a1.im + b1.im};
    v[4] = {a1.re - b1.re, a1.im - b1.im};
    v[2] = {a2.re + b2.re, a2.im + b2.im};
    v[3] = {a2.re - b2.re, a2.im - b2.im};
}

template <typename T>
__device__ __forceinline__ void dft8(Cx<T>* v, T dir) {
    const T r2 = T(0.70710678118654752440);
    Cx<T> e[4] = {v[0], v[2], v[4], v[6]};
    Cx<T> o[4] = {v[1], v[3], v[5], v[7]};
    dft4(e, dir);
    dft4(o, dir);
    // w8^k = exp(dir * 2 pi i k / 8)
    Cx<T> w1 = {r2, dir * r2};
    Cx<T> w3 = {-r2, dir * r2};
    Cx<T> o1 = cmul(o[1], w1);
    Cx<T> o2 = mul_di(o[2], dir);
    Cx<T> o3 = cmul(o[3], w3);
    v[0] = {e[0].re + o[0].re, e[0].im + o[0].im};
    v[4] = {e[0].re - o[0].re, e[0].im - o[0].im};
    v[1] = {e[1].re + o1.re, e[1].im + o1.im};
    v[5] = {e[1].re - o1.re, e[1].im - o1.im};
    v[2] = {e[2].re + o2.re, e[2].im + o2.im};
    v[6] = {e[2].re - o2.re, e[2].im - o2.im};
    v[3] = {e[3].re + o3.re, e[3].im + o3.im};
    v[7] = {e[3].re - o3.re, e[3].im - o3.im};
}

template <int R, typename T>
__device__ __forceinline__ void dft(Cx<T>* v, T dir) {
    if constexpr (R == 2) dft2(v);
    else if constexpr (R == 3) dft3(v, dir);
    else if constexpr (R == 4) dft4(v, dir);
    else if constexpr (R == 5) dft5(v, dir);
    else dft8(v, dir);
}

// Exact quotient and remainder of small non-negative integers (x < 2^22, d >= 1) through a
// float reciprocal rd = 1/d and one correction step: a few VALU ops instead of the ~25 of a
// generic 32-bit division.
__device__ __forceinline__ int udiv_small(int x, int d, float rd, int& rem) {
    int q = (int)((float)x * rd);
    int r = x - q * d;
    if (r < 0) {
        --q;
        r += d;
    } else if (r >= d) {
        ++q;
        r -= d;
    }
    rem = r;
    return q;
}

// What separates the passes of an in-place FFT: the workgroup's barrier, or, when one wave owns
// all its rows (WAVE), only an order for the compiler to keep (a wave's LDS operations complete in
// order).
template <bool WAVE>
__device__ __forceinline__ void fft_sync() {
    if constexpr (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// Butterflies of radix R that a thread holds in one pass: what fits 8 complex registers. With one
// butterfly per thread whatever the radix, a tile was as narrow as its plan's smallest radix left it
// (half-length 120 = 8 * 5 * 3: 8 pencils, 150 with a 2: 4), and rows of 64 or 32 bytes ran the
// transforms at half the rate or less: along y at 256 x 128 cells per plane, forward and inverse, 240 2.04 ->
// 3.38 and 2.29 -> 3.21 TB/s, 300 1.33 -> 2.90 and 1.56 -> 2.97, 180 1.62 -> 2.73 and 1.73 -> 2.45; along x2
// alike (300 1.59 -> 3.00 both ways).
__host__ __device__ constexpr int fft_hold(int R) { return R >= 5 ? 1 : 8 / R; }

// One run-time pass of radix R over P sequences of length n = nb*R, span Ns (cfft_lds_ip).
template <typename T, bool WAVE, int R>
__device__ __forceinline__ void cfft_pass_rt(T* __restrict__ xr, T* __restrict__ xi, int ld, int P, int n, int Ns,
                                             const T* twr, const T* twi, T dir, int tid, int nthr) {
    constexpr int U = fft_hold(R);
    const int nb = n / R, tstep = nb / Ns, tasks = P * nb;
    const float rnb = 1.0f / (float)nb, rNs = 1.0f / (float)Ns;
    Cx<T> v[U][R];
    int orow[U], ob[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = tid + u * nthr;
        if (t < tasks) {
            int jj, k;
            orow[u] = udiv_small(t, nb, rnb, jj) * ld;
            const int blk = udiv_small(jj, Ns, rNs, k);
            ob[u] = blk * Ns * R + k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = orow[u] + pidx(jj + r * nb);
                v[u][r] = {xr[o], xi[o]};
            }
            if (Ns > 1) {
                int w = 0;
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    w += k * tstep;
                    // table holds exp(-2 pi i t/n); forward (dir=-1) uses it as is, inverse conj
                    v[u][r] = cmul(v[u][r], Cx<T>{twr[w], (dir < 0) ? twi[w] : -twi[w]});
                }
            }
            dft<R>(v[u], dir);
        }
    }
    fft_sync<WAVE>();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (tid + u * nthr < tasks) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = orow[u] + pidx(ob[u] + r * Ns);
                xr[o] = v[u][r].re;
                xi[o] = v[u][r].im;
            }
        }
    }
    fft_sync<WAVE>();
}

// In-place complex FFT of P sequences of length fp.n held in ONE buffer (split re/im, row
// stride ld). Each radix pass: every thread loads its butterflies (fft_hold of them at most: 8
// complex values), the workgroup synchronises, then every thread stores. Needs
// P * n <= R * fft_hold(R) * nthr for every radix R of the plan (fft_tile_ok). The caller
// synchronises before (data ready); the result is visible on return. WAVE: tid is the lane of the
// one wave that owns the P sequences, nthr = 64.
template <typename T, bool WAVE = false>
__device__ void cfft_lds_ip(T* __restrict__ xr, T* __restrict__ xi, int ld, int P, const FftPlan& fp,
                            const T* twr, const T* twi, T dir, int tid, int nthr) {
    int Ns = 1;
    for (int p = 0; p < fp.count; ++p) {
        const int R = fp.rad[p];
        // opaque: nothing of a pass is hoisted out of the loop over them, where the values of all
        // radices would hold registers together
        int t = tid;
        asm volatile("" : "+v"(t));
        switch (R) {
            case 2: cfft_pass_rt<T, WAVE, 2>(xr, xi, ld, P, fp.n, Ns, twr, twi, dir, t, nthr); break;
            case 3: cfft_pass_rt<T, WAVE, 3>(xr, xi, ld, P, fp.n, Ns, twr, twi, dir, t, nthr); break;
            case 4: cfft_pass_rt<T, WAVE, 4>(xr, xi, ld, P, fp.n, Ns, twr, twi, dir, t, nthr); break;
            case 5: cfft_pass_rt<T, WAVE, 5>(xr, xi, ld, P, fp.n, Ns, twr, twi, dir, t, nthr); break;
            default: cfft_pass_rt<T, WAVE, 8>(xr, xi, ld, P, fp.n, Ns, twr, twi, dir, t, nthr); break;
        }
        Ns *= R;
    }
}

// ------------------------------------------------------------------ compile-time radix plans
// The same in-place passes with the length and the radices fixed at compile time, for the plans that
// radix_plan makes of n = 16 ... 512 and of n = 24, 48, 96, 192 (periodic lengths and x2 counts of
// 48 to 384) with radices up to 8. With n, R and the span Ns constants, the butterfly's pencil,
// block and twiddle indices are shifts and masks (or one constant product), and where the strides are
// multiples of 8 or do not carry into the padding every LDS address of a butterfly is one computed
// base plus constant offsets: pidx(base + r*s) equals pidx(base) + r*s + (r*s >> 3) whenever
// s % 8 == 0, or when base is a multiple of 8 and r*s < 8, so the offsets fold into the LDS
// instructions. 768 x 384 x 256, whose x2 transforms have n = 192: 0.350 -> 0.289 ms forward and 0.367 ->
// 0.296 inverse over the run-time passes; projections of 192 x 192 x 96 0.167 -> 0.149 ms.
__device__ __forceinline__ constexpr int poff(int x) { return x + (x >> 3); }

template <typename T, bool WAVE, int n, int R, int Ns>
__device__ __forceinline__ void cfft_pass_static(T* __restrict__ xr, T* __restrict__ xi, int ld, int P,
                                                 const T* twr, const T* twi, T dir, int tid, int nthr) {
    constexpr int nb = n / R;
    constexpr int tstep = n / (Ns * R);
    // loads at jj + r*nb: whole padding steps apart, or jj < nb <= 8 a power of two (no carry)
    constexpr bool lin_load = nb % 8 == 0 || 8 % nb == 0;
    // stores at blk*Ns*R + k + r*Ns, k < Ns
    constexpr bool lin_store = Ns % 8 == 0 || (8 % Ns == 0 && ((Ns * R) % 8 == 0 || 8 % (Ns * R) == 0));
    // powers of two take one butterfly per thread: their tiles fill the workgroup so
    constexpr int U = (n & (n - 1)) == 0 ? 1 : fft_hold(R);
    Cx<T> v[U][R];
    int orow[U], ob[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int t = tid + u * nthr;
        if (t < P * nb) {
            const int pen = t / nb;  // constants: shifts and masks for powers of two
            const int jj = t - pen * nb;
            const int blk = jj / Ns;
            const int k = jj - blk * Ns;
            orow[u] = pen * ld;
            const int ia = orow[u] + pidx(jj);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = lin_load ? ia + poff(r * nb) : orow[u] + pidx(jj + r * nb);
                v[u][r] = {xr[o], xi[o]};
            }
            if (Ns > 1) {
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    const int w = k * (r * tstep);
                    // table holds exp(-2 pi i t/n); forward (dir=-1) uses it as is, inverse conj
                    v[u][r] = cmul(v[u][r], Cx<T>{twr[w], (dir < 0) ? twi[w] : -twi[w]});
                }
            }
            dft<R>(v[u], dir);
            ob[u] = blk * Ns * R + k;
        }
    }
    fft_sync<WAVE>();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if (tid + u * nthr < P * nb) {
            const int oa = orow[u] + pidx(ob[u]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = lin_store ? oa + poff(r * Ns) : orow[u] + pidx(ob[u] + r * Ns);
                xr[o] = v[u][r].re;
                xi[o] = v[u][r].im;
            }
        }
    }
    fft_sync<WAVE>();
}

template <typename T, bool WAVE, int n, int Ns, int R, int... Rest>
__device__ __forceinline__ void cfft_passes_static(T* xr, T* xi, int ld, int P, const T* twr, const T* twi, T dir,
                                                   int tid, int nthr) {
    cfft_pass_static<T, WAVE, n, R, Ns>(xr, xi, ld, P, twr, twi, dir, tid, nthr);
    if constexpr (sizeof...(Rest) > 0) cfft_passes_static<T, WAVE, n, Ns * R, Rest...>(xr, xi, ld, P, twr, twi, dir, tid, nthr);
}

// cfft_lds_ip with the plans listed above taken by the compile-time passes (fp.fixed, which the plan
// sets), every other plan by the run-time passes. Same contract. One switch on the length: its compares
// lie together, where a chain of tests would step over each body on the way to the next and wait for
// its instructions (a small kernel is bound by that).
template <typename T, bool WAVE = false>
__device__ __forceinline__ void cfft_lds(T* __restrict__ xr, T* __restrict__ xi, int ld, int P, const FftPlan& fp,
                                         const T* twr, const T* twi, T dir, int tid, int nthr) {
    switch (fp.fixed) {
        case 16: cfft_passes_static<T, WAVE, 16, 1, 4, 4>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 24: cfft_passes_static<T, WAVE, 24, 1, 8, 3>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 32: cfft_passes_static<T, WAVE, 32, 1, 8, 4>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 48: cfft_passes_static<T, WAVE, 48, 1, 4, 4, 3>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 64: cfft_passes_static<T, WAVE, 64, 1, 8, 8>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 96: cfft_passes_static<T, WAVE, 96, 1, 8, 4, 3>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 128: cfft_passes_static<T, WAVE, 128, 1, 8, 4, 4>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 192: cfft_passes_static<T, WAVE, 192, 1, 8, 8, 3>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 256: cfft_passes_static<T, WAVE, 256, 1, 8, 8, 4>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        case 512: cfft_passes_static<T, WAVE, 512, 1, 8, 8, 8>(xr, xi, ld, P, twr, twi, dir, tid, nthr); break;
        default: cfft_lds_ip<T, WAVE>(xr, xi, ld, P, fp, twr, twi, dir, tid, nthr);
    }
}

// Whether the compile-time passes of cfft_lds take the plan: its length, else 0.
inline int fixed_plan(const FftPlan& fp) {
    auto is = [&](std::initializer_list<int> rad) {
        return fp.count == (int)rad.size() && std::equal(rad.begin(), rad.end(), fp.rad);
    };
    const bool listed = (fp.n == 16 && is({4, 4})) || (fp.n == 24 && is({8, 3})) || (fp.n == 32 && is({8, 4})) ||
                        (fp.n == 48 && is({4, 4, 3})) || (fp.n == 64 && is({8, 8})) || (fp.n == 96 && is({8, 4, 3})) ||
                        (fp.n == 128 && is({8, 4, 4})) || (fp.n == 192 && is({8, 8, 3})) ||
                        (fp.n == 256 && is({8, 8, 4})) || (fp.n == 512 && is({8, 8, 8}));
    return listed ? fp.n : 0;
}

// Smallest radix of a plan (bounds the butterflies per pass of cfft_lds_ip).
__host__ __device__ inline int min_radix(const FftPlan& fp) {
    int r = 8;
    for (int p = 0; p < fp.count; ++p) r = fp.rad[p] < r ? fp.rad[p] : r;
    return fp.count ? r : 8;
}

// Whether nthr threads hold P sequences of the plan in one pass of each radix (powers of two at one
// butterfly per thread: theirs are compile-time passes, whose 16 pencils need no more).
inline bool fft_tile_ok(const FftPlan& fp, long P, int nthr) {
    const bool pow2 = (fp.n & (fp.n - 1)) == 0;
    for (int p = 0; p < fp.count; ++p)
        if (P * fp.n > (long)fp.rad[p] * (pow2 ? 1 : fft_hold(fp.rad[p])) * nthr) return false;
    return true;
}

// Workgroup size of the transform kernels: 512 threads hold 16 pencils of a length-256 real
// transform in one pass, so every HBM row access of a tile covers a full 128-byte line.
constexpr int kFftThreads = 512;

}  // namespace eddy
