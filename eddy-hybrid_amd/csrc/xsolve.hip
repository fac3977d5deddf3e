// xsolve.hip -- the x1 tridiagonal solves of every (y-mode j, x2-mode m) line.
//
// After the y-FFT and the x2 transform, DIRECT's per-mode 2-D problem (direct.f:788-797)
// separates into one tridiagonal system per line:
//   AM(i) x(i-1) + (BM(i) - AK_j / RP(i+1)^2 + lam_m) x(i) + CM(i) x(i+1) = d(i),
// with AM(1) = CM(M) = 0 (Neumann walls, direct.f:344-352). The singular line (j = 0, null
// x2 mode) is pinned with x(1) = 0, as the reference's IPRES=3 branch pins its singular mode
// (direct.f:849-852); the plain-mean removal of direct.f:895-898 follows in the inverse x2
// transform.
//
// Algorithm (per line, P threads, Q = M/P rows each, Q >= 3): every thread eliminates its
// own chunk with a modified Thomas sweep that expresses each row through the chunk's first
// and last unknowns; the 2P chunk-end unknowns form a tridiagonal system solved by parallel
// cyclic reduction across the P lanes of the line (wave shuffles); each thread then
// back-substitutes its chunk. A wave stages the elements of its 64/P lines, which are contiguous
// in S, through LDS of its own, so that global reads and writes are contiguous and no workgroup
// barrier is needed.
//
// What bounds it: FP64 instruction issue beside HBM (16 B per cell). A wave's 64/P lines are 64 Q
// elements, so lane and element index differ by multiples of 64: the staging addresses are one
// base plus constants, where indexing a padded 2-D tile took a quotient per element each way.
// 512 x 256 x 256 FP64 (P = 64, Q = 8): 0.153 -> 0.127 ms, 4.2 TB/s; the production grid's 1024-row
// x2 lines (P = 64, Q = 16): 0.231 -> 0.169 ms.
#include <algorithm>
#include <numeric>
#include <type_traits>

#include "batch_device.h"
#include "kernels.h"
#include "stencil_device.h"

namespace eddy {

// Reciprocal from the hardware estimate and Newton steps (within about an ulp): the pivots
// of the eliminations are far from zero and denormals, so the scaling steps of a correctly
// rounded division buy nothing here.
__device__ __forceinline__ double fast_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    double e = __builtin_fma(-x, r, 1.0);
    r = __builtin_fma(r, e, r);
    e = __builtin_fma(-x, r, 1.0);
    return __builtin_fma(r, e, r);
}
__device__ __forceinline__ float fast_rcp(float x) {
    float r = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(r, __builtin_fmaf(-x, r, 1.0f), r);
}

// Lane permute of a 32- or 64-bit value by a precomputed byte address (4 * source lane).
__device__ __forceinline__ float lane_get(float v, int addr) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}
__device__ __forceinline__ double lane_get(double v, int addr) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_ds_bpermute(addr, (int)b);
    const int hi = __builtin_amdgcn_ds_bpermute(addr, (int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

template <typename T>
struct XArgs {
    T* S;
    T* linesum;
    Dims d;
    Tables<T> tb;
    int P, Q;
    long lbeg, lend;  // line range (j-major lines j*N + m) of this launch
    // periodic lines (the CYC kernels): row 0 couples to x(M-1) through beta (AM(1)) and row
    // M-1 to x(0) through alpha (CM(M)); the tables hold 0 in those two slots
    T alpha, beta;
};

// LDS elements of a wave's 64 Q staged values (index e at e + e/8: a lane's Q consecutive values
// and the staging's 64 consecutive ones both spread over the banks)
__host__ __device__ inline int xlds_wave(int Q) { return 72 * Q + 2; }

// A coupling to a chunk end this small no longer reaches a result (2^-80 of its neighbour): the
// even unknowns are decoupled and the remaining reduction steps would return them unchanged.
// Each step squares the couplings, so on most lines (those of all but the lowest wavenumbers)
// two or three of the log2 P steps are left over.
constexpr double kDecoupled = 0x1p-80;

// Solve the wave's 64/P lines, P lanes and Q rows per lane (FIXED: Q = QMAX and M = P*Q, no row
// checks). get(r) is the right-hand side of this lane's row r, put(r, x) takes its solution.
// Returns the sum of the lane's solution rows. CYC: periodic lines, solved as the tridiagonal
// part T' plus a rank-one correction (Sherman-Morrison, the method of the reference's CYCLIC,
// numrec.f:754-781): T = T' + u v^T with u = (g, 0, ..., 0, alpha), v = (1, 0, ..., 0, beta/g),
// g = -b(0); the elimination carries the second right-hand side u beside d, and
// x = y - z (y_0 + beta y_{M-1}/g) / (1 + z_0 + beta z_{M-1}/g). The singular line is pinned at
// x(0) = 0 and solved without the correction (its corner couplings act on x(0) = 0).
template <typename T, int QMAX, bool FIXED, bool CYC, typename Get, typename Put>
__device__ __forceinline__ T xsolve_lines(const XArgs<T>& a, int p, int lane, T akj, T lam, bool pin, Get get,
                                          Put put) {
    const int P = a.P, Q = FIXED ? QMAX : a.Q, M = a.d.M;
    // periodic line: the corrected diagonals of rows 0 and M-1 and the second right-hand side
    const bool cyc = CYC && !pin;
    const T g = CYC ? -(a.tb.bm[0] - akj * a.tb.r2inv[0] + lam) : T(0);

    T aa[QMAX], cc[QMAX], dd[QMAX];
    T ee[CYC ? QMAX : 1];
    const int ib = p * Q;
    // rows in batches of 4 whose coefficients (tables in thread order: row p*Q + r at r*P + p) are
    // loaded together; rows past M are identity rows of the tables with a zero right-hand side
    constexpr int B = QMAX < 4 ? QMAX : 4;
#pragma unroll
    for (int r0 = 0; r0 < QMAX; r0 += B) {
        T ta[B], tc[B], tb[B], tr[B], td[B];
#pragma unroll
        for (int u = 0; u < B && r0 + u < QMAX; ++u) {
            const int r = FIXED ? r0 + u : min(r0 + u, Q - 1);
            const unsigned o = (unsigned)sizeof(T) * (unsigned)(r * P + p);
            ta[u] = ld_off(a.tb.am, o);
            tc[u] = ld_off(a.tb.cm, o);
            tb[u] = ld_off(a.tb.bm, o);
            tr[u] = ld_off(a.tb.r2inv, o);
            td[u] = get(r);
        }
#pragma unroll
        for (int u = 0; u < B && r0 + u < QMAX; ++u) {
            const int r = r0 + u;
            if (!FIXED && r >= Q) continue;
            T av = ta[u], cv = tc[u], bv = tb[u] - akj * tr[u] + lam;
            T dv = (FIXED || ib + r < M) ? td[u] : T(0);
            if (r == 0) {  // the singular line: x(0) = 0
                const bool z = pin && p == 0;
                av = z ? T(0) : av;
                bv = z ? T(1) : bv;
                cv = z ? T(0) : cv;
                dv = z ? T(0) : dv;
            }
            T ev = T(0);
            if (CYC && cyc) {
                if (ib + r == 0) {
                    bv = bv - g;
                    ev = g;
                }
                if (ib + r == M - 1) {
                    bv = bv - a.alpha * a.beta / g;
                    ev = a.alpha;
                }
            }
            if (r < 2) {
                const T inv = fast_rcp(bv);
                aa[r] = av * inv;
                cc[r] = cv * inv;
                dd[r] = dv * inv;
                if constexpr (CYC) ee[r] = ev * inv;
            } else {
                const T inv = fast_rcp(bv - av * cc[r - 1]);
                dd[r] = (dv - av * dd[r - 1]) * inv;
                if constexpr (CYC) ee[r] = (ev - av * ee[r - 1]) * inv;
                aa[r] = -av * aa[r - 1] * inv;
                cc[r] = cv * inv;
            }
        }
    }
#pragma unroll
    for (int r = QMAX - 3; r >= 1; --r) {
        if (r <= Q - 3) {
            dd[r] -= cc[r] * dd[r + 1];
            if constexpr (CYC) ee[r] -= cc[r] * ee[r + 1];
            aa[r] -= cc[r] * aa[r + 1];
            cc[r] = -cc[r] * cc[r + 1];
        }
    }
    {
        const T inv = fast_rcp(T(1) - cc[0] * aa[1]);
        dd[0] = (dd[0] - cc[0] * dd[1]) * inv;
        if constexpr (CYC) ee[0] = (ee[0] - cc[0] * ee[1]) * inv;
        aa[0] = aa[0] * inv;
        cc[0] = -cc[0] * cc[1] * inv;
    }
    // reduced system: rows 2p (chunk first) and 2p+1 (chunk last)
    T lastA = T(0), lastC = T(0), lastD = T(0), lastE = T(0);
#pragma unroll
    for (int r = 0; r < QMAX; ++r)
        if (r == Q - 1) {
            lastA = aa[r];
            lastC = cc[r];
            lastD = dd[r];
            if constexpr (CYC) lastE = ee[r];
        }
    // The 2P chunk-end unknowns y (y_2p = chunk p's first row, y_2p+1 its last) form a
    // tridiagonal system with unit diagonal: lane p holds rows 2p (a0, c0, d0) and 2p+1
    // (a1, c1, d1). One cyclic-reduction step removes the odd unknowns from the even rows;
    // the P even unknowns are then solved by parallel cyclic reduction across the lanes
    // (wave shuffles), and each odd unknown follows from its own row:
    // y_2p+1 = d1 - a1 y_2p - c1 y_2p+2. Rows at a line end have the coupling to the missing
    // side at exactly 0 (AM(1) = CM(M) = 0 at the walls, identity padding rows), so the
    // neighbours fetched across a line end (wrapping inside the wave) are finite values
    // multiplied by 0.
    T a0 = aa[0], c0 = cc[0], d0 = dd[0], e0 = CYC ? ee[0] : T(0);
    const T a1 = lastA, c1 = lastC, d1 = lastD, e1 = lastE;
    {  // even row 2p minus a0 * row 2p-1 (lane p-1's odd row) minus c0 * row 2p+1 (own odd row)
        const int up = ((lane - 1) & 63) << 2;
        const T ua = lane_get(a1, up), uc = lane_get(c1, up), ud = lane_get(d1, up);
        const T i0 = fast_rcp(T(1) - a0 * uc - c0 * a1);
        const T na0 = -a0 * ua * i0, nc0 = -c0 * c1 * i0, nd0 = (d0 - a0 * ud - c0 * d1) * i0;
        if constexpr (CYC) e0 = (e0 - a0 * lane_get(e1, up) - c0 * e1) * i0;
        a0 = na0;
        c0 = nc0;
        d0 = nd0;
    }
    for (int dl = 1; dl < P; dl <<= 1) {  // even rows at distance dl lanes
        if (!__any(fabs(a0) > T(kDecoupled) || fabs(c0) > T(kDecoupled))) break;
        const int up = ((lane - dl) & 63) << 2, dn = ((lane + dl) & 63) << 2;
        const T ua = lane_get(a0, up), uc = lane_get(c0, up), ud = lane_get(d0, up);
        const T va = lane_get(a0, dn), vc = lane_get(c0, dn), vd = lane_get(d0, dn);
        const T i0 = fast_rcp(T(1) - a0 * uc - c0 * va);
        const T na0 = -a0 * ua * i0, nc0 = -c0 * vc * i0, nd0 = (d0 - a0 * ud - c0 * vd) * i0;
        if constexpr (CYC) e0 = (e0 - a0 * lane_get(e0, up) - c0 * lane_get(e0, dn)) * i0;
        a0 = na0;
        c0 = nc0;
        d0 = nd0;
    }
    const T x0 = d0;
    const T xl = d1 - a1 * x0 - c1 * lane_get(x0, ((lane + 1) & 63) << 2);
    // periodic line: the correction factor from y_0, z_0 (lane p = 0, row 0) and y_{M-1},
    // z_{M-1} (lane (M-1)/Q, row (M-1) mod Q) of the line's lanes
    T fact = T(0), z0 = T(0), zl = T(0);
    if constexpr (CYC) {
        z0 = e0;
        zl = e1 - a1 * z0 - c1 * lane_get(z0, ((lane + 1) & 63) << 2);
        const int pl1 = (M - 1) / Q, rl1 = (M - 1) - pl1 * Q;
        T yM = T(0), zM = T(0);
#pragma unroll
        for (int r = 0; r < QMAX; ++r)
            if (r == rl1) {
                yM = (r == 0) ? x0 : ((r == Q - 1) ? xl : dd[r] - aa[r] * x0 - cc[r] * xl);
                zM = (r == 0) ? z0 : ((r == Q - 1) ? zl : ee[r] - aa[r] * z0 - cc[r] * zl);
            }
        const int first = lane - p;  // the line's lanes are consecutive within the wave
        const T y0l = lane_get(x0, first << 2), z0l = lane_get(z0, first << 2);
        yM = lane_get(yM, (first + pl1) << 2);
        zM = lane_get(zM, (first + pl1) << 2);
        if (cyc) fact = (y0l + a.beta * yM / g) / (T(1) + z0l + a.beta * zM / g);
    }
    // back-substitute (own rows only), accumulate the line sum
    T part = T(0);
#pragma unroll
    for (int r = 0; r < QMAX; ++r) {
        if (FIXED || r < Q) {
            T x;
            if (r == 0) x = x0;
            else if (r == Q - 1) x = xl;
            else x = dd[r] - aa[r] * x0 - cc[r] * xl;
            if constexpr (CYC) {
                T z;
                if (r == 0) z = z0;
                else if (r == Q - 1) z = zl;
                else z = ee[r] - aa[r] * z0 - cc[r] * zl;
                x -= fact * z;
            }
            put(r, x);
            part += x;
        }
    }
    return part;
}

// One block of 256/P lines (logical line block `lb`), 64/P lines per wave.
template <typename T, int QMAX, bool FIXED, bool CYC = false>
__device__ __forceinline__ void xsolve_tile(const XArgs<T>& a, int lb) {
    extern __shared__ unsigned char smem_raw[];
    const Dims d = a.d;
    const int P = a.P, Q = FIXED ? QMAX : a.Q, M = d.M, N = d.N;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int LW = 64 / P;  // lines per wave
    T* const tile = reinterpret_cast<T*>(smem_raw) + w * xlds_wave(Q);
    // line numbers and element offsets in 32 bits: S holds fewer than 2^29 elements (the plan
    // rejects fields of 4 GiB and more)
    const int line0 = (int)a.lbeg + (lb * 4 + w) * LW;
    const int nl = min(LW, (int)a.lend - line0);  // the wave's lines
    if (nl <= 0) return;

    // The wave's lines, contiguous in S, into its LDS: element lane + 64 u, every load in flight
    // together; elements past the last line read the last one (finite values for lanes whose
    // results are not stored)
    T* const blk = a.S + (size_t)line0 * (size_t)M;
    const int nel = nl * M;
    const int wi = lane + (lane >> 3);
    {
        T v[QMAX];
        if (nel == 64 * QMAX) {  // wave-uniform
#pragma unroll
            for (int u = 0; u < QMAX; ++u) v[u] = blk[lane + 64 * u];
        } else {
#pragma unroll
            for (int u = 0; u < QMAX; ++u)
                v[u] = ld_off(blk, (unsigned)sizeof(T) * (unsigned)min(lane + 64 * u, nel - 1));
        }
#pragma unroll
        for (int u = 0; u < QMAX; ++u)
            if (FIXED || u < Q) tile[wi + 72 * u] = v[u];
    }
    // the wave's LDS operations complete in order; this only keeps the compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

    const int lw = lane / P, p = lane - lw * P;
    const int l = line0 + min(lw, nl - 1);
    int j, m;
    if (LW <= N) {  // one quotient for the wave
        const int j0 = line0 / N;
        m = line0 - j0 * N + (l - line0);
        j = j0;
        if (m >= N) {
            m -= N;
            ++j;
        }
    } else {
        j = l / N;
        m = l - j * N;
    }
    const T akj = a.tb.akj[j];
    const T lam = a.tb.lamj ? a.tb.lamj[l] : a.tb.lam[m];
    const bool pin = j == 0 && m == d.null_m;
    // the lane's rows: elements e0 + r of the wave's region
    const int e0 = FIXED ? lane * QMAX : lw * M + p * Q;
    auto at = [&](int r) { return e0 + r + ((e0 + r) >> 3); };
    T part = xsolve_lines<T, QMAX, FIXED, CYC>(
        a, p, lane, akj, lam, pin,
        [&](int r) { return tile[FIXED ? at(r) : min(at(r), xlds_wave(Q) - 1)]; },
        [&](int r, T x) {
            if (FIXED || p * Q + r < M) tile[at(r)] = x;
        });
    if (j == 0) {
        // reduce over the P lanes of this line (consecutive lanes of one wave, P <= 64)
        for (int off = P >> 1; off > 0; off >>= 1) part += __shfl_xor(part, off, 64);
        if (lw < nl && p == 0) a.linesum[m] = part;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (nel == 64 * QMAX) {
#pragma unroll
        for (int u = 0; u < QMAX; ++u) blk[lane + 64 * u] = tile[wi + 72 * u];
    } else {
#pragma unroll
        for (int u = 0; u < QMAX; ++u)
            if (lane + 64 * u < nel) st_off(blk, (unsigned)sizeof(T) * (unsigned)(lane + 64 * u), tile[wi + 72 * u]);
    }
}

// The lines are walked from the last to the first, against the order of the x2 transforms on both
// sides: each then starts on what the pass before it left in the 256 MiB memory-side cache. At
// 768 x 384 x 256 (a spectrum of 604 MB) this solve takes 0.284 ms instead of 0.310 and the inverse
// x2 transform 0.369 instead of 0.387; nothing changes at 512 x 256 x 256 (268 MB) and below.
template <typename T, int QMAX, bool FIXED, bool CYC>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && FIXED ? (QMAX <= 8 ? 6 : 4) : 1)))
k_xsolve(XArgs<T> a) {
    xsolve_tile<T, QMAX, FIXED, CYC>(a, xcd_tile(gridDim.x - 1 - blockIdx.x, gridDim.x));
}

// Pick P (threads per line, a power of two <= 64) and Q (rows per thread, 3 <= Q <= qmax):
// an exact split M = P*Q when one exists, else Q = ceil(M/P) with the line padded by
// P*Q - M identity rows (CM(M) = 0 at the wall decouples them, so they solve to 0). Lines
// up to 64 x 32 = 2048 rows.
static bool pick_pq(int M, int qmax, int& P, int& Q) {
    for (P = 1; P <= 64; P <<= 1) {
        if (M % P) continue;
        Q = M / P;
        if (Q >= 3 && Q <= qmax) return true;
    }
    for (P = 1; P <= 64; P <<= 1) {
        Q = std::max(3, (M + P - 1) / P);
        if (Q <= qmax) return true;
    }
    return false;
}

static bool pick_pq_any(int M, int chunk, int& P, int& Q) {
    // the largest kernel template holds kXsolveMaxChunk rows per thread
    const int qmax = chunk > 0 ? std::min(chunk, kXsolveMaxChunk) : 16;
    return pick_pq(M, qmax, P, Q) || pick_pq(M, 16, P, Q) || pick_pq(M, 32, P, Q);
}

bool xsolve_partition(int M, int chunk, int& P, int& Q) { return pick_pq_any(M, chunk, P, Q); }

// Kernel template of a line length: the exact splits M = P*Q with Q of the usual grids have their
// own (kFixed + Q: no row checks, constant LDS offsets), every other split runs the smallest
// template of at least Q rows.
constexpr int kFixed = 64;
static int xsolve_class(int M, int P, int Q, bool cyc) {
    if (!cyc && P * Q == M && (Q == 6 || Q == 8 || Q == 10 || Q == 12 || Q == 16)) return kFixed + Q;
    return Q <= 4 ? 4 : (Q <= 8 ? 8 : (Q <= 16 ? 16 : 32));
}

// go(integral QMAX, FIXED) of a class
template <typename Go>
static void xsolve_dispatch(int cls, Go go) {
    switch (cls) {
        case kFixed + 6: go(std::integral_constant<int, 6>{}, std::true_type{}); break;
        case kFixed + 8: go(std::integral_constant<int, 8>{}, std::true_type{}); break;
        case kFixed + 10: go(std::integral_constant<int, 10>{}, std::true_type{}); break;
        case kFixed + 12: go(std::integral_constant<int, 12>{}, std::true_type{}); break;
        case kFixed + 16: go(std::integral_constant<int, 16>{}, std::true_type{}); break;
        case 4: go(std::integral_constant<int, 4>{}, std::false_type{}); break;
        case 8: go(std::integral_constant<int, 8>{}, std::false_type{}); break;
        case 16: go(std::integral_constant<int, 16>{}, std::false_type{}); break;
        default: go(std::integral_constant<int, 32>{}, std::false_type{}); break;
    }
}

template <typename T>
int launch_xsolve(hipStream_t st, const Dims& d, const Tables<T>& tb, T* S, T* linesum, int chunk, int j0, int nj,
                  int cyc, double alpha, double beta) {
    XArgs<T> a{};
    a.S = S;
    a.linesum = linesum;
    a.d = d;
    a.tb = tb;
    a.alpha = T(alpha);
    a.beta = T(beta);
    int P = 0, Q = 0;
    if (!pick_pq_any(d.M, chunk, P, Q)) return -1;
    a.P = P;
    a.Q = Q;
    const int LPW = 256 / P;
    a.lbeg = (long)j0 * d.N;
    a.lend = (long)(j0 + nj) * d.N;
    const long nlines = a.lend - a.lbeg;
    dim3 grid((unsigned)((nlines + LPW - 1) / LPW));
    const size_t sh = 4 * (size_t)xlds_wave(Q) * sizeof(T);
    xsolve_dispatch(xsolve_class(d.M, P, Q, cyc != 0), [&](auto qmax, auto fixed) {
        auto go = [&](auto fn) {
            (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
            hipLaunchKernelGGL(fn, grid, dim3(256), sh, st, a);
        };
        if constexpr (decltype(fixed)::value) go(k_xsolve<T, decltype(qmax)::value, true, false>);
        else if (cyc) go(k_xsolve<T, decltype(qmax)::value, false, true>);
        else go(k_xsolve<T, decltype(qmax)::value, false, false>);
    });
    return 0;
}

// ------------------------------------------------------------------ batched (one item per workgroup)
// One kernel per rows-per-thread template: a kernel holding every template would take the
// registers of the largest (QMAX = 32) for all problems.
// Bounds where the unbounded kernel sits just above an occupancy step (8 rows: 86 VGPRs, 6 waves
// per SIMD at 80; 16 rows: 148, 4 waves at 128).
template <typename T, int QMAX, bool FIXED>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && FIXED ? (QMAX <= 8 ? 6 : 4) : 1)))
k_batch_xsolve(const Job<XArgs<T>>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total, [](const Job<XArgs<T>>& J, int t) { xsolve_tile<T, QMAX, FIXED>(J.a, t); });
}

template <typename T>
int prepare_xsolve(const std::vector<BatchProblem<T>>& pr, StageLaunch& out, std::vector<void*>& owned) {
    struct Item {
        int idx, P, Q, cls;
    };
    std::vector<Item> items;
    for (int idx = 0; idx < (int)pr.size(); ++idx) {
        int P = 0, Q = 0;
        if (!pick_pq_any(pr[idx].d.M, pr[idx].chunk, P, Q)) return -2;
        items.push_back({idx, P, Q, xsolve_class(pr[idx].d.M, P, Q, false)});
    }
    auto lds_of = [&](const Item& it) { return 4 * (size_t)xlds_wave(it.Q) * sizeof(T); };
    // grouped by template class (most rows first); the tiles of most LDS first, then the
    // longest x1 lines
    std::stable_sort(items.begin(), items.end(), [&](const Item& x, const Item& y) {
        if (x.cls % kFixed != y.cls % kFixed) return x.cls % kFixed > y.cls % kFixed;
        if (x.cls != y.cls) return x.cls > y.cls;
        const int ox = lds_occupancy(lds_of(x)), oy = lds_occupancy(lds_of(y));
        return ox != oy ? ox < oy : pr[x.idx].d.M > pr[y.idx].d.M;
    });
    std::vector<Job<XArgs<T>>> jobs;
    out = StageLaunch{};
    for (const Item& it : items) {
        const BatchProblem<T>& p = pr[it.idx];
        Job<XArgs<T>> j{};
        XArgs<T>& a = j.a;
        a.S = p.S;
        a.linesum = p.linesum;
        a.d = p.d;
        a.tb = p.tb;
        a.P = it.P;
        a.Q = it.Q;
        a.lbeg = 0;
        a.lend = (long)p.d.L * p.d.N;
        const int LPW = 256 / it.P;
        j.ntx = 1;
        j.ntiles = (int)(((long)p.d.L * p.d.N + LPW - 1) / LPW);
        j.aux = it.cls;
        if (!add_class_job(out, jobs, j, it.cls, lds_of(it))) return -1;
    }
    return upload_jobs(jobs, out, owned);
}

template <typename T>
void batch_xsolve(hipStream_t st, const StageLaunch& sl) {
    for (int c = 0; c < sl.ncls; ++c) {
        xsolve_dispatch(sl.cls_q[c], [&](auto qmax, auto fixed) {
            auto fn = k_batch_xsolve<T, decltype(qmax)::value, decltype(fixed)::value>;
            const size_t lds = sl.cls_lds[c];
            (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            const int total = sl.cls_total[c];
            const Job<XArgs<T>>* jobs = (const Job<XArgs<T>>*)sl.jobs + sl.cls_job[c];
            hipLaunchKernelGGL(fn, dim3(std::max(total, 1)), dim3(256), lds, st, jobs, sl.cls_job[c + 1] - sl.cls_job[c],
                               total);
        });
    }
}

template int prepare_xsolve<double>(const std::vector<BatchProblem<double>>&, StageLaunch&, std::vector<void*>&);
template int prepare_xsolve<float>(const std::vector<BatchProblem<float>>&, StageLaunch&, std::vector<void*>&);
template void batch_xsolve<double>(hipStream_t, const StageLaunch&);
template void batch_xsolve<float>(hipStream_t, const StageLaunch&);

template int launch_xsolve<double>(hipStream_t, const Dims&, const Tables<double>&, double*, double*, int, int, int,
                                   int, double, double);
template int launch_xsolve<float>(hipStream_t, const Dims&, const Tables<float>&, float*, float*, int, int, int, int,
                                  double, double);

}  // namespace eddy
