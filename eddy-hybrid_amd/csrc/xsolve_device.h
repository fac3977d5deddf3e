// xsolve_device.h -- the tridiagonal line solve of one wave (64/P lines, P lanes per line), shared by
// the line-solve kernels (xsolve.hip) and the fused plane kernel (zplane.hip). The algorithm is
// described in xsolve.hip.
#pragma once

#include <type_traits>

#include "common.h"
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

// How a line-solve template takes its rows: any Q <= QMAX; Q = QMAX with lines that end in padding
// (M <= P*Q); Q = QMAX and M = P*Q (no row checks).
enum XRows { XR_ANY = 0, XR_PADDED = 1, XR_EXACT = 2 };

// Solve the wave's 64/P lines, P lanes and Q rows per lane. get(r) is the right-hand side of this lane's
// row r (any finite value in lanes without a line), put(r, x) takes its solution. Returns the sum of
// the lane's solution rows. CYC: periodic lines, solved as the tridiagonal part T' plus a rank-one
// correction (Sherman-Morrison, the method of the reference's CYCLIC, numrec.f:754-781):
// T = T' + u v^T with u = (g, 0, ..., 0, alpha), v = (1, 0, ..., 0, beta/g), g = -b(0); the
// elimination carries the second right-hand side u beside d, and
// x = y - z (y_0 + beta y_{M-1}/g) / (1 + z_0 + beta z_{M-1}/g). The singular line is pinned at
// x(0) = 0 and solved without the correction (its corner couplings act on x(0) = 0).
template <typename T, int QMAX, int ROWS, bool CYC, typename Get, typename Put>
__device__ __forceinline__ T xsolve_lines(const XArgs<T>& a, int p, int lane, T akj, T lam, bool pin, Get get,
                                          Put put) {
    constexpr bool FIXED = ROWS != XR_ANY;
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
            T dv = (ROWS == XR_EXACT || ib + r < M) ? td[u] : T(0);
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
    // neighbours fetched across a line end (wrapping inside the wave) are multiplied by 0; they are
    // finite in lanes without a line too, as get() is (0 * NaN would be NaN).
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

// Kernel template of a line length: the exact splits M = P*Q with Q of the usual grids have their
// own (kExact + Q: no row checks), as have the other splits into 7 to 12 rows (all that the default
// partition makes of M > 96; kPadded + Q: constant loops, the lines staged at P*Q elements each so that LDS
// offsets are constant too); every other split runs the smallest template of at least Q rows. At
// 128 x 128 lines, against the next larger of 8 or 16 rows with its row checks: 300 rows 2.27 -> 2.87 TB/s,
// 350 2.62 -> 3.21, 528 2.45 -> 3.29, 576 2.58 -> 3.60, 700 3.04 -> 3.84, 200 2.31 -> 2.44, 450 3.10 -> 3.19. P < 16
// (M <= 96) has 8 lines and more to a wave, whose staging would look their bounds up one by one.
constexpr int kExact = 64, kPadded = 128;
inline int xsolve_class(int M, int P, int Q, bool cyc) {
    if (!cyc && P * Q == M && (Q == 6 || Q == 8 || Q == 10 || Q == 12 || Q == 16)) return kExact + Q;
    if (!cyc && P >= 16 && Q >= 7 && Q <= 12) return kPadded + Q;
    return Q <= 4 ? 4 : (Q <= 8 ? 8 : (Q <= 16 ? 16 : 32));
}

template <int QMAX, int ROWS, typename Go>
void xsolve_go(Go go) {
    go(std::integral_constant<int, QMAX>{}, std::integral_constant<int, ROWS>{});
}

// go(integral QMAX, integral XRows) of a class
template <typename Go>
void xsolve_dispatch(int cls, Go go) {
    switch (cls) {
        case kExact + 6: xsolve_go<6, XR_EXACT>(go); break;
        case kExact + 8: xsolve_go<8, XR_EXACT>(go); break;
        case kExact + 10: xsolve_go<10, XR_EXACT>(go); break;
        case kExact + 12: xsolve_go<12, XR_EXACT>(go); break;
        case kExact + 16: xsolve_go<16, XR_EXACT>(go); break;
        case kPadded + 7: xsolve_go<7, XR_PADDED>(go); break;
        case kPadded + 8: xsolve_go<8, XR_PADDED>(go); break;
        case kPadded + 9: xsolve_go<9, XR_PADDED>(go); break;
        case kPadded + 10: xsolve_go<10, XR_PADDED>(go); break;
        case kPadded + 11: xsolve_go<11, XR_PADDED>(go); break;
        case kPadded + 12: xsolve_go<12, XR_PADDED>(go); break;
        case 4: xsolve_go<4, XR_ANY>(go); break;
        case 8: xsolve_go<8, XR_ANY>(go); break;
        case 16: xsolve_go<16, XR_ANY>(go); break;
        default: xsolve_go<32, XR_ANY>(go); break;
    }
}

}  // namespace eddy
