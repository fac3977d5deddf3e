// stencil.hip -- the HBM-streaming FP64 kernels around the solve:
//   DIVERGENCE (timeindeg.f:944-946) fused with the DP/ALFXDT scaling (Eddy6.f:2715) and,
//     optionally, the volume-weighted solvability sums;
//   CORRECT (timeindeg.f:1002, 1012, 1022) over the faces of setup.f:17-72;
//   the 7-point operator of DIRECT (for residuals), the final mean removal + ghost fill of
//   the defect correction, and reductions.
// Element-wise kernels: one thread per interior cell, x1 fastest, 64 x1 cells by 4 y rows
// per block. Reducing kernels: a block owns 64 x1 cells of one x2 plane for every y (its
// threads stride over y), so a whole plane row reduces to one partial per block.
#include <algorithm>
#include <numeric>

#include "batch_device.h"
#include "kernels.h"
#include "reduce_device.h"
#include "stencil_device.h"

namespace eddy {

static inline dim3 cell_grid(const Dims& d) { return dim3(ceil_div(d.M, 64), ceil_div(d.L, 4), d.N); }
static inline dim3 red_grid(const Dims& d) { return dim3(ceil_div(d.M, 64), 1, d.N); }
static const dim3 kCellBlock(64, 4, 1);

int reduce_blocks(const Dims& d) { return ceil_div(d.M, 64) * d.N; }

// logical (x, y, z) block of an XCD-ordered 3-D grid
struct Blk {
    int x, y, z;
};
__device__ __forceinline__ Blk xcd_block() {
    const int gx = gridDim.x, gy = gridDim.y;
    const int t = xcd_tile(blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z), gx * gy * gridDim.z);
    return Blk{t % gx, (t / gx) % gy, t / (gx * gy)};
}

__global__ void __launch_bounds__(256) k_divergence(Dims d, Metrics mt, const double* __restrict__ us,
                                                    const double* __restrict__ vs, const double* __restrict__ ws,
                                                    double* __restrict__ div, double scale, double* part,
                                                    int accumulate, const double* __restrict__ dscale) {
    const Blk bk = xcd_block();
    if (dscale) scale = dscale[1];
    const int i = bk.x * 64 + threadIdx.x;
    const int k = bk.z;
    double vb = 0.0;
    if (i < d.M) {
        const int I = i + 1, K = k + 1;
        for (int j = threadIdx.y; j < d.L; j += 4) {
            const double v = div_at(d, mt, us, vs, ws, i, j, k) * scale;
            div[sidx(d, I, j + 1, K)] = v;
            if (accumulate) vb += cell_vol(mt, i, j, k) * v;
        }
    }
    if (accumulate) block_partial<RED_OP_SUM>(vb, part, linear_bid());
}

// CORRECT along memory instead of along rows: the interior rows J = 1..L of a plane are one span
// of L*nx consecutive elements, cut into blocks of 512 * kSpanParts elements that start on a
// 128-byte line (when the bases do), two neighbouring elements per lane and part. Every access of
// the six velocity fields and of dp is then a whole aligned 1 KiB per wave, where a 64-cell block of
// a row (nx = M + 2 elements, starting one past a ghost) straddles five lines with partial lines at
// both ends, read and written by two blocks. The ghosts inside the span (4 of nx) are loaded and
// not stored. Fields and rows of any alignment take the same 16-byte accesses (d2u). HBM bound;
// with the streamed velocities and the block order below 0.398 -> 0.343 ms at 512 x 256 x 256,
// 0.493 -> 0.407 ms at 302 x 130 x 1026, 0.058 -> 0.044 ms at 300 x 128 x 128.
constexpr int kSpanParts = 2;
constexpr int kSpan = 512 * kSpanParts;  // elements per block

typedef double d2 __attribute__((ext_vector_type(2)));
// a pair at any element: rows of odd nx and fields that start between two 16-byte boundaries are
// read and written with the same 16-byte instructions, which need dword alignment only
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

struct CorrArgs {
    Dims d;
    Metrics mt;
    const double *us, *vs, *ws;
    double *uo, *vo, *wo;
    const double* dp;
    unsigned rnx;  // row_reciprocal(nx)
};

static inline unsigned row_magic(const Dims& d) { return row_reciprocal(d.nx); }

// Blocks of a plane's span (its start rounded down to 16 elements).
__host__ __device__ inline int span_blocks(const Dims& d) { return ceil_div(d.L * d.nx + 15, kSpan); }

__device__ __forceinline__ d2 ld_pair(const double* b, unsigned off) {
    return *reinterpret_cast<const d2u*>(reinterpret_cast<const char*>(b) + off);
}
// The velocities are streamed (read once, written once): non-temporal, so that they do not push dp's
// planes out of L2 nor the solve's arrays out of the memory-side cache. Small fields (kCorrectCached) are
// read through the caches: the forward y transform has just read u*, and what it left there is lost to a
// non-temporal load (projections on the same fields again, and on others each time, read past the caches and
// through them: 128 x 96 x 64 0.0540 -> 0.0501 ms and 0.0558 -> 0.0548, 120 x 90 x 80 0.0704 -> 0.0661 and 0.0723 ->
// 0.0715; CORRECT alone 0.0109 -> 0.0072 and 0.0126 -> 0.0137 at the first). Larger fields gain in the second case
// what they lose in the first (203 x 101 x 90 0.1091 -> 0.1029 and 0.1112 -> 0.1121; its four calls of a substep
// 0.131 -> 0.136; 240 x 128 x 128 0.1418 -> 0.1339 and 0.1474 -> 0.1578) and stay streamed; CORRECT alone on the same
// fields again is then slower than through the caches (128 x 128 x 128 0.0235 and 0.0197), on others faster (0.0249
// and 0.0279).
template <bool STREAM>
__device__ __forceinline__ d2 ld_velocity(const double* b, unsigned off) {
    const d2u* p = reinterpret_cast<const d2u*>(reinterpret_cast<const char*>(b) + off);
    if constexpr (STREAM) return __builtin_nontemporal_load(p);
    else return *p;
}
__device__ __forceinline__ void st_stream(double* b, unsigned off, d2 v) {
    __builtin_nontemporal_store(v, reinterpret_cast<d2u*>(reinterpret_cast<char*>(b) + off));
}

__device__ __forceinline__ Pair span_pair(const Dims& d, unsigned r, unsigned rnx) {
    return plane_pair(d.nx, d.M, d.L, r, rnx);
}

// Whether the seven fields of CORRECT exceed `mib` MiB together.
static inline bool correct_exceeds(size_t cells, size_t mib) { return 7 * sizeof(double) * cells > (mib << 20); }
constexpr size_t kCorrectCached = 64;  // MiB up to which the velocities are read through the caches

// Block `b` of plane k's span (k 0-based interior).
template <bool STREAM>
__device__ __forceinline__ void correct_span(const CorrArgs& c, double alfxdt, int refresh, int k, int b, int tid) {
    const Dims& d = c.d;
    const unsigned nx = (unsigned)d.nx, pl = nx * (unsigned)d.ny;
    const unsigned plane = pl * (unsigned)(k + 1);
    const unsigned e0 = ((plane + nx) & ~15u) + (unsigned)b * kSpan + 2u * (unsigned)tid;
    const double cwK = c.mt.cw[k + 1];
    const bool wface = k + 1 <= d.nz - 3 + d.cyc_z;
    const int ulast = d.nx - 3 + d.cyc_x, vlast = d.ny - 2 - d.ycopy;
    unsigned o[kSpanParts];
    Pair pr[kSpanParts];
    d2 p0[kSpanParts], u[kSpanParts], v[kSpanParts], w[kSpanParts], pn[kSpanParts], pt[kSpanParts];
    double pe[kSpanParts];
#pragma unroll
    for (int q = 0; q < kSpanParts; ++q) {
        pr[q] = span_pair(d, e0 + 512u * q - plane, c.rnx);
        o[q] = 8u * (pr[q].on ? e0 + 512u * q : plane + nx);
        p0[q] = ld_pair(c.dp, o[q]);
        pe[q] = ld_off(c.dp, o[q] + 16u);
        pn[q] = ld_pair(c.dp, o[q] + 8u * nx);
        pt[q] = ld_pair(c.dp, o[q] + 8u * pl);
        u[q] = ld_velocity<STREAM>(c.us, o[q]);
        v[q] = ld_velocity<STREAM>(c.vs, o[q]);
        w[q] = ld_velocity<STREAM>(c.ws, o[q]);
    }
#pragma unroll
    for (int q = 0; q < kSpanParts; ++q) {
        if (!pr[q].on) continue;
        const int i = pr[q].i, j = pr[q].j;
        const int i1 = min(i + 1, d.nx - 1);
        const double bvJ = c.mt.bv[j];
        d2 un, vn, wn;
        un.x = u[q].x - c.mt.au[i] * (p0[q].y - p0[q].x) * alfxdt;
        un.y = u[q].y - c.mt.au[i1] * (pe[q] - p0[q].y) * alfxdt;
        const double gx = bvJ * (pn[q].x - p0[q].x) * alfxdt, gy = bvJ * (pn[q].y - p0[q].y) * alfxdt;
        vn.x = v[q].x - (c.mt.cart ? gx : gx / c.mt.rp[i]);
        vn.y = v[q].y - (c.mt.cart ? gy : gy / c.mt.rp[i1]);
        wn.x = w[q].x - cwK * (pt[q].x - p0[q].x) * alfxdt;
        wn.y = w[q].y - cwK * (pt[q].y - p0[q].y) * alfxdt;
        const bool a0 = i >= 1, a1 = i + 1 <= d.M;  // the pair's interior cells
        const bool u0 = a0 && i <= ulast, u1 = a1 && i + 1 <= ulast;
        const bool vf = j <= vlast;
        auto put = [&](double* f, unsigned at, d2 x, bool s0, bool s1) {
            if (s0 && s1) st_stream(f, at, x);
            else if (s0) st_off(f, at, x.x);
            else if (s1) st_off(f, at + 8u, x.y);
        };
        if (a0 && a1 && u0 && u1) {
            st_stream(c.uo, o[q], un);
            if (vf) st_stream(c.vo, o[q], vn);
            if (wface) st_stream(c.wo, o[q], wn);
        } else {
            put(c.uo, o[q], un, u0, u1);
            if (vf) put(c.vo, o[q], vn, a0, a1);
            if (wface) put(c.wo, o[q], wn, a0, a1);
        }
        // periodic y ghost rows of the corrected faces (the velocity BC step after CORRECT,
        // Eddy6.f:2746-2761): row J=1 mirrors J=NY-1, row J=NY mirrors J=2
        if (refresh && !d.ycopy && (j == 1 || j == d.L)) {
            const unsigned g = o[q] + (j == d.L ? 0u - 8u * nx * (unsigned)(d.ny - 2) : 8u * nx * (unsigned)(d.ny - 2));
            put(c.uo, g, un, u0, u1);
            if (vf) put(c.vo, g, vn, a0, a1);
            if (wface) put(c.wo, g, wn, a0, a1);
        }
    }
}

// Item t of a problem's nb x N blocks, the planes in pairs (dp's plane k + 1, read with plane k, is
// then read again by the block after it).
template <bool STREAM>
__device__ __forceinline__ void correct_item(const CorrArgs& c, double alfxdt, int refresh, int t, int nb) {
    const int c0 = t / (2 * nb), r = t - c0 * 2 * nb, kc = min(2, c.d.N - 2 * c0);
    const int b = r / kc;
    correct_span<STREAM>(c, alfxdt, refresh, 2 * c0 + r - b * kc, b, (int)threadIdx.x);
}

// The XCDs share the field in runs of kCorrectRun blocks, so that the eight of them work within a
// window of it, once the fields exceed the 256 MiB memory-side cache: 0.392 -> 0.343 ms at
// 512 x 256 x 256 (5.5 TB/s of 56 B/cell; runs of 2 to 64 within 2 %) and 0.457 -> 0.415 ms at
// 302 x 130 x 1026 over one contiguous eighth per XCD, which ties up 56 far-apart streams. Smaller
// fields come out of the cache and take the eighths (256 x 128 x 128: 0.0385 against 0.0397 ms).
constexpr int kCorrectRun = 16;

template <bool STREAM>
__global__ void __launch_bounds__(256) k_correct_span(CorrArgs c, double alfxdt, int refresh, int runs,
                                                      const double* __restrict__ dscale) {
    const int b = blockIdx.x, n = gridDim.x;
    if (dscale) alfxdt = dscale[0];
    const int t = runs ? xcd_run(b, n, kCorrectRun) : xcd_tile(b, n);
    correct_item<STREAM>(c, alfxdt, refresh, t, n / c.d.N);
}

static CorrArgs corr_args(const Dims& d, const Metrics& mt, const double* us, const double* vs, const double* ws,
                          double* uo, double* vo, double* wo, const double* dp) {
    return CorrArgs{d, mt, us, vs, ws, uo, vo, wo, dp, row_magic(d)};
}

// SCRINFO's divergence range over the same spans (fmin / fmax as the reference's MIN / MAX). A block
// takes the spans b, b + nbx, ... of `planes` consecutive planes and keeps w of the plane below
// in registers on its way up, so that w is read once but for the lowest plane's neighbour. It leaves its
// minimum at part[slot], its maximum at part[nb + slot]. 24 B/cell, HBM bound: 0.430 -> 0.360 ms at
// 768 x 384 x 256 over a kernel of row blocks, and one fold instead of two and a log kernel after it. The x1
// metrics are read once per span: inside the plane loop they were waited for behind the cells' branches, plane by
// plane (whole calls at 768 x 384 x 256 0.367 -> 0.336 ms, 512 x 256 x 256 0.191 -> 0.166, 256 x 192 x 96 on the same
// fields again 0.050 -> 0.045, where the row blocks had taken 0.046).
__global__ void __launch_bounds__(256) k_div_minmax(Dims d, Metrics mt, const double* __restrict__ us,
                                                    const double* __restrict__ vs, const double* __restrict__ ws,
                                                    double* part, unsigned rnx, int nbx, int planes, int runs) {
    const int nb = gridDim.x;
    const int t = runs ? xcd_run(blockIdx.x, nb, kCorrectRun) : xcd_tile(blockIdx.x, nb);
    const int kg = t / nbx, k0 = kg * planes, k1 = min(k0 + planes, d.N);
    const unsigned nx = (unsigned)d.nx, pl = nx * (unsigned)d.ny, nspan = (unsigned)span_blocks(d);
    double mn = 1e300, mx = -1e300;
    for (unsigned b = (unsigned)(t - kg * nbx); b < nspan; b += (unsigned)nbx) {
        // the span's elements of the group's first plane; the others' are whole planes above
        Pair pr[kSpanParts];
        unsigned o[kSpanParts];
        d2 wm[kSpanParts], api[kSpanParts];
        double bpj[kSpanParts];
#pragma unroll
        for (int q = 0; q < kSpanParts; ++q) {
            const unsigned r = (nx & ~15u) + b * kSpan + 512u * q + 2u * threadIdx.x;
            pr[q] = span_pair(d, r, rnx);
            o[q] = 8u * ((pr[q].on ? r : nx) + pl * (unsigned)(k0 + 1));
            bpj[q] = mt.bp[pr[q].on ? pr[q].j : 1];
            const int i = pr[q].on ? pr[q].i : 0;
            api[q].x = mt.ap[i];
            api[q].y = mt.ap[i + 1];
            wm[q] = ld_pair(ws, o[q] - 8u * pl);
        }
        for (int k = k0; k < k1; ++k) {
            const double cpk = mt.cp[k + 1];
            d2 u[kSpanParts], v[kSpanParts], vm[kSpanParts], w[kSpanParts];
            double um[kSpanParts];
#pragma unroll
            for (int q = 0; q < kSpanParts; ++q) {
                u[q] = ld_pair(us, o[q]);
                um[q] = ld_off(us, o[q] - 8u);
                v[q] = ld_pair(vs, o[q]);
                vm[q] = ld_pair(vs, o[q] - 8u * nx);
                w[q] = ld_pair(ws, o[q]);
            }
#pragma unroll
            for (int q = 0; q < kSpanParts; ++q) {
                // div_at's arithmetic
                auto one = [&](int I, double ap, double um1, double u1, double vm1, double v1, double wm1, double w1) {
                    if (!pr[q].on || I < 1 || I > d.M) return;
                    const double c = cpk * (w1 - wm1);
                    double x;
                    if (mt.cart) {
                        x = ap * (u1 - um1) + bpj[q] * (v1 - vm1) + c;
                    } else {
                        const double rpi = mt.rp[I];
                        x = ap * (mt.ru[I] * u1 - mt.ru[I - 1] * um1) / rpi + bpj[q] * (v1 - vm1) / rpi + c;
                    }
                    mn = fmin(mn, x);
                    mx = fmax(mx, x);
                };
                one(pr[q].i, api[q].x, um[q], u[q].x, vm[q].x, v[q].x, wm[q].x, w[q].x);
                one(pr[q].i + 1, api[q].y, u[q].x, u[q].y, vm[q].y, v[q].y, wm[q].y, w[q].y);
                wm[q] = w[q];
                o[q] += 8u * pl;
            }
        }
    }
    block_partial<RED_OP_MIN>(mn, part, (int)blockIdx.x);
    block_partial<RED_OP_MAX>(mx, part + nb, (int)blockIdx.x);
}

// red[RED_DMIN], red[RED_DMAX] from the n block minima and maxima of k_div_minmax, one workgroup of
// 1024 threads; with a log, the step's epilogue too: log[2 s], log[2 s + 1] for s = *step < cap, then
// *step = s + 1.
__global__ void __launch_bounds__(1024) k_fold_minmax(const double* __restrict__ part, int n, double* red, double* log,
                                                      int* step, int cap) {
    double mn = 1e300, mx = -1e300;
#pragma unroll 8
    for (int t = threadIdx.x; t < n; t += 1024) {
        mn = fmin(mn, part[t]);
        mx = fmax(mx, part[n + t]);
    }
    __shared__ double w[2][16];
    mn = wave_min(mn);
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) {
        w[0][threadIdx.x >> 6] = mn;
        w[1][threadIdx.x >> 6] = mx;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 16; ++q) {
            mn = fmin(mn, w[0][q]);
            mx = fmax(mx, w[1][q]);
        }
        red[RED_DMIN] = mn;
        red[RED_DMAX] = mx;
        if (log) {
            const int s = step[0];
            if (s >= 0 && s < cap) {
                log[2 * s] = mn;
                log[2 * s + 1] = mx;
            }
            step[0] = s + 1;
        }
    }
}

__global__ void __launch_bounds__(256) k_laplacian(Dims d, Op64 op, const double* __restrict__ phi,
                                                   double* __restrict__ out) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int j = bk.y * 4 + threadIdx.y;
    const int k = bk.z;
    if (i >= d.M || j >= d.L) return;
    out[sidx(d, i + 1, j + 1, k + 1)] = lap_at(d, op, phi, i, j, k);
}

// Partial sums over the interior of (rhs - L(phi))^2.
__global__ void __launch_bounds__(256) k_resid_sumsq(Dims d, Op64 op, const double* __restrict__ phi,
                                                     const double* __restrict__ rhs, double* part) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int k = bk.z;
    double rr = 0.0;
    if (i < d.M) {
        for (int j = threadIdx.y; j < d.L; j += 4) {
            const double r = rhs[sidx(d, i + 1, j + 1, k + 1)] - lap_at(d, op, phi, i, j, k);
            rr += r * r;
        }
    }
    block_partial<RED_OP_SUM>(rr, part, linear_bid());
}

// phi <- phi - mean (mean = red[RED_PHISUM]/(M L N)) on the interior, then the ghosts as
// direct.f:1035-1106 leaves them: x ghosts copies (MP=1) or periodic images (MP=0), y ghosts
// periodic images (LP=0) or copies (LP=1), z ghost planes zero.
__global__ void __launch_bounds__(256) k_shift_ghosts(Dims d, double* __restrict__ phi, const double* red) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int j = bk.y * 4 + threadIdx.y;
    const int k = bk.z;
    if (i >= d.M || j >= d.L) return;
    const double mean = red[RED_PHISUM] / ((double)d.M * (double)d.L * (double)d.N);
    const int I = i + 1, J = j + 1, K = k + 1;
    const double v = phi[sidx(d, I, J, K)] - mean;
    int Is[3], Js[3];
    int ni = 0, nj = 0;
    Is[ni++] = I;
    if (i == (d.cyc_x ? d.M - 1 : 0)) Is[ni++] = 0;
    if (i == (d.cyc_x ? 0 : d.M - 1)) Is[ni++] = d.nx - 1;
    Js[nj++] = J;
    if (j == (d.ycopy ? 0 : d.L - 1)) Js[nj++] = 0;
    if (j == (d.ycopy ? d.L - 1 : 0)) Js[nj++] = d.ny - 1;
    for (int p = 0; p < ni; ++p)
        for (int q = 0; q < nj; ++q) phi[sidx(d, Is[p], Js[q], K)] = v;
    if (k == 0 || k == d.N - 1) {
        const int Kg = (k == 0) ? 0 : d.nz - 1;
        for (int p = 0; p < ni; ++p)
            for (int q = 0; q < nj; ++q) phi[sidx(d, Is[p], Js[q], Kg)] = 0.0;
    }
}

__global__ void __launch_bounds__(256) k_sumsq(Dims d, const double* __restrict__ a, double* part) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int k = bk.z;
    double s = 0.0;
    if (i < d.M) {
        for (int j = threadIdx.y; j < d.L; j += 4) {
            const double v = a[sidx(d, i + 1, j + 1, k + 1)];
            s += v * v;
        }
    }
    block_partial<RED_OP_SUM>(s, part, linear_bid());
}

// The RHS check: sum vol*b and sum vol*|b| over the finite interior values of b, and the count
// of non-finite ones, as three per-block partials (nb blocks each).
__global__ void __launch_bounds__(256) k_rhs_check(Dims d, Metrics mt, const double* __restrict__ b, double* part,
                                                   int nb) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int k = bk.z;
    double s = 0.0, sa = 0.0, nf = 0.0;
    if (i < d.M) {
        for (int j = threadIdx.y; j < d.L; j += 4) {
            const double v = b[sidx(d, i + 1, j + 1, k + 1)];
            if (!isfinite(v)) {
                nf += 1.0;
                continue;
            }
            const double vol = cell_vol(mt, i, j, k);
            s += vol * v;
            sa += vol * fabs(v);
        }
    }
    block_partial<RED_OP_SUM>(s, part, linear_bid());
    block_partial<RED_OP_SUM>(sa, part + nb, linear_bid());
    block_partial<RED_OP_SUM>(nf, part + 2 * nb, linear_bid());
}

// dst <- src - red[RED_VOLB]/red[RED_VOL] on the interior (volume-weighted solvability
// shift of the RHS).
__global__ void __launch_bounds__(256) k_copy_shift(Dims d, const double* __restrict__ src,
                                                    double* __restrict__ dst, const double* red) {
    const Blk bk = xcd_block();
    const int i = bk.x * 64 + threadIdx.x;
    const int j = bk.y * 4 + threadIdx.y;
    const int k = bk.z;
    if (i >= d.M || j >= d.L) return;
    const double c = red[RED_VOLB] / red[RED_VOL];
    const size_t o = sidx(d, i + 1, j + 1, k + 1);
    dst[o] = src[o] - c;
}

// REFRESHBC (refreshbc.f:1-28) on one GPU: the z ghost planes exchanged with the
// neighbouring slabs. With x2 walls both neighbours are walls and the ghosts stay as DIRECT
// left them (zero); with a periodic x2 (ITYPE(5) = ITYPE(6) = 500) the one slab is its own
// neighbour: DP(:,:,1) = DP(:,:,NZ-1), DP(:,:,NZ) = DP(:,:,2).
__global__ void k_refresh_z(Dims d, double* __restrict__ dp) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t pl = (size_t)d.nx * d.ny;
    if (t >= pl) return;
    dp[t] = dp[t + pl * (size_t)(d.nz - 2)];
    dp[t + pl * (size_t)(d.nz - 1)] = dp[t + pl];
}

__global__ void k_fill(double* p, size_t n, double v) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = v;
}

// out[b] = the sum of part[b*n .. b*n + n) for workgroup b of 1024 threads; out[1] = next where next is
// not 0 (one workgroup).
__global__ void __launch_bounds__(1024) k_fold(const double* __restrict__ part, int n, double* out, double next) {
    part += (size_t)blockIdx.x * n;
    double v = 0.0;
#pragma unroll 8
    for (int t = threadIdx.x; t < n; t += 1024) v += part[t];
    __shared__ double w[16];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = w[0];
        for (int q = 1; q < 16; ++q) s += w[q];
        out[blockIdx.x] = s;
        if (next != 0.0) out[1] = next;
    }
}

// ------------------------------------------------------------------ batched (one item per workgroup)
struct CellArgs {
    Dims d;
    double* dp;
    double* rhs;
    const double* red;
};

constexpr int kCellRows = 4;  // y rows per thread of a batch cell item

// One item: 64 x1 cells by 4 * kCellRows y rows of one x2 plane, threads 64 x 4 with rows
// j0, j0 + 4, ... each; items run x1 block fastest, then the y block, then the plane (ntx x1
// blocks, nty y blocks per plane). Every load of a thread is issued before its first store:
// rows past L load a clamped in-range row and store nothing. (One row per thread left the
// per-item set-up, the job search and argument loads, on every 256 cells: the copy stages
// ran 1.3-1.9x slower.)
template <int OP>
__device__ __forceinline__ void cell_tile(const CellArgs& c, int t, int ntx, int nty) {
    constexpr int R = kCellRows;
    const Dims& d = c.d;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int xb = t % ntx, r = t / ntx;
    const int i = xb * 64 + tx;
    const int j0 = (r % nty) * (4 * R) + ty;
    const int k = r / nty;
    if (i >= d.M) return;
    const int I = i + 1, K = k + 1;
    size_t o[R];
#pragma unroll
    for (int q = 0; q < R; ++q) o[q] = sidx(d, I, min(j0 + 4 * q, d.L - 1) + 1, K);
    if (OP == BC_COPY_RHS) {
        double x[R];
#pragma unroll
        for (int q = 0; q < R; ++q) x[q] = c.dp[o[q]];
#pragma unroll
        for (int q = 0; q < R; ++q)
            if (j0 + 4 * q < d.L) c.rhs[o[q]] = x[q];
    } else {
        const double mean = c.red[RED_PHISUM] / ((double)d.M * (double)d.L * (double)d.N);
        double x[R];
#pragma unroll
        for (int q = 0; q < R; ++q) x[q] = c.dp[o[q]];
#pragma unroll
        for (int q = 0; q < R; ++q) {
            const int j = j0 + 4 * q;
            if (j >= d.L) continue;
            const int J = j + 1;
            const double v = x[q] - mean;
            int Is[3], Js[3];
            int ni = 0, nj = 0;
            Is[ni++] = I;
            if (i == 0) Is[ni++] = 0;
            if (i == d.M - 1) Is[ni++] = d.nx - 1;
            Js[nj++] = J;
            if (j == d.L - 1) Js[nj++] = 0;
            if (j == 0) Js[nj++] = d.ny - 1;
            for (int p = 0; p < ni; ++p)
                for (int qq = 0; qq < nj; ++qq) c.dp[sidx(d, Is[p], Js[qq], K)] = v;
            if (k == 0 || k == d.N - 1) {
                const int Kg = (k == 0) ? 0 : d.nz - 1;
                for (int p = 0; p < ni; ++p)
                    for (int qq = 0; qq < nj; ++qq) c.dp[sidx(d, Is[p], Js[qq], Kg)] = 0.0;
            }
        }
    }
}

template <int OP>
__global__ void __launch_bounds__(256) k_batch_cells(const Job<CellArgs>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total, [](const Job<CellArgs>& J, int t) { cell_tile<OP>(J.a, t, J.ntx, J.aux); });
}

// CORRECT of a batch; alf = {ALFXDT, 1/ALFXDT} on the device.
template <bool STREAM>
__global__ void __launch_bounds__(256) k_batch_correct(const Job<CorrArgs>* jobs, int njobs, int total,
                                                       const double* __restrict__ alf) {
    const double alfxdt = alf[0];
    run_item<kCorrectRun>(jobs, njobs, total,
                          [=](const Job<CorrArgs>& J, int t) { correct_item<STREAM>(J.a, alfxdt, 1, t, J.ntx); });
}

template <typename T>
static int prepare_cells_t(const std::vector<BatchProblem<T>>& pr, int op, StageLaunch& out,
                           std::vector<void*>& owned) {
    std::vector<int> order(pr.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return pr[x].d.L > pr[y].d.L; });
    std::vector<Job<CellArgs>> jobs;
    int total = 0;
    for (int idx : order) {
        const BatchProblem<T>& p = pr[idx];
        Job<CellArgs> j{};
        CellArgs& c = j.a;
        c.d = p.d;
        c.dp = p.dp;
        c.rhs = const_cast<double*>(p.rhs);
        c.red = p.red;
        j.ntx = ceil_div(p.d.M, 64);
        j.aux = ceil_div(p.d.L, 4 * kCellRows);  // y blocks per plane
        j.ntiles = j.ntx * j.aux * p.d.N;
        j.first = total;
        total += j.ntiles;
        jobs.push_back(j);
    }
    void* buf = nullptr;
    if (hipMalloc(&buf, jobs.size() * sizeof(jobs[0])) != hipSuccess) return -1;
    owned.push_back(buf);
    if (hipMemcpy(buf, jobs.data(), jobs.size() * sizeof(jobs[0]), hipMemcpyHostToDevice) != hipSuccess) return -1;
    out.jobs = buf;
    out.njobs = (int)jobs.size();
    out.total = total;
    out.lds = 0;
    return 0;
}

int prepare_cells(const std::vector<BatchProblem<double>>& pr, int op, StageLaunch& out, std::vector<void*>& owned) {
    if (op != BC_CORRECT) return prepare_cells_t(pr, op, out, owned);
    std::vector<Job<CorrArgs>> jobs;
    out = StageLaunch{};
    size_t cells = 0;
    for (const auto& p : pr) {
        cells += (size_t)p.d.nx * p.d.ny * p.d.nz;
        Job<CorrArgs> j{};
        j.a = corr_args(p.d, p.mt, p.us, p.vs, p.ws, p.uo, p.vo, p.wo, p.dp);
        j.ntx = span_blocks(p.d);
        j.ntiles = j.ntx * p.d.N;
        if (!add_class_job(out, jobs, j, 0, 0)) return -1;
    }
    out.alf = pr.empty() ? nullptr : pr[0].dscale;
    out.kind = correct_exceeds(cells, kCorrectCached);
    return upload_jobs(jobs, out, owned);
}
int prepare_cells_f(const std::vector<BatchProblem<float>>& pr, int op, StageLaunch& out,
                    std::vector<void*>& owned) {
    return prepare_cells_t(pr, op, out, owned);
}

void batch_cells(hipStream_t st, const StageLaunch& sl, int op) {
    if (op == BC_CORRECT) {
        auto go = [&](auto fn) {
            hipLaunchKernelGGL(fn, dim3(std::max(sl.total, 1)), dim3(256), 0, st, (const Job<CorrArgs>*)sl.jobs,
                               sl.njobs, sl.total, sl.alf);
        };
        if (sl.kind) go(k_batch_correct<true>);
        else go(k_batch_correct<false>);
        return;
    }
    auto go = [&](auto fn) {
        hipLaunchKernelGGL(fn, dim3(std::max(sl.total, 1)), dim3(256), 0, st, (const Job<CellArgs>*)sl.jobs, sl.njobs,
                           sl.total);
    };
    if (op == BC_COPY_RHS) go(k_batch_cells<BC_COPY_RHS>);
    else go(k_batch_cells<BC_SHIFT_GHOSTS>);
}

__global__ void __launch_bounds__(1024) k_batch_fold(const FoldJob* jobs) {
    const FoldJob J = jobs[blockIdx.x];
    double v = (J.op == RED_OP_SUM) ? 0.0 : ((J.op == RED_OP_MIN) ? 1e300 : -1e300);
    for (int t = threadIdx.x; t < J.n; t += blockDim.x) {
        const double x = J.part[t];
        v = (J.op == RED_OP_SUM) ? v + x : ((J.op == RED_OP_MIN) ? fmin(v, x) : fmax(v, x));
    }
    __shared__ double w[16];
    if (J.op == RED_OP_SUM) v = wave_reduce<RED_OP_SUM>(v);
    else if (J.op == RED_OP_MIN) v = wave_reduce<RED_OP_MIN>(v);
    else v = wave_reduce<RED_OP_MAX>(v);
    if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = w[0];
        for (int q = 1; q < (int)(blockDim.x >> 6); ++q)
            s = (J.op == RED_OP_SUM) ? s + w[q] : ((J.op == RED_OP_MIN) ? fmin(s, w[q]) : fmax(s, w[q]));
        *J.out = s;
    }
}

void batch_fold(hipStream_t st, const FoldJob* jobs, int njobs) {
    if (njobs > 0) hipLaunchKernelGGL(k_batch_fold, dim3(njobs), dim3(1024), 0, st, jobs);
}

void launch_fold(hipStream_t st, const double* part, int n, double* out, int count, double next) {
    hipLaunchKernelGGL(k_fold, dim3(count), dim3(1024), 0, st, part, n, out, next);
}

void launch_divergence(hipStream_t st, const Dims& d, const Metrics& mt, const double* us, const double* vs,
                       const double* ws, double* div, double scale, const Reduce& rd, int accumulate_compat,
                       const double* dscale) {
    hipLaunchKernelGGL(k_divergence, red_grid(d), kCellBlock, 0, st, d, mt, us, vs, ws, div, scale, rd.part,
                       accumulate_compat, dscale);
    if (accumulate_compat) {
        const int nb = reduce_blocks(d);
        launch_fold(st, rd.part, nb, rd.red + RED_VOLB, 1, mt.vol_total);
    }
}

void launch_div_minmax(hipStream_t st, const Dims& d, const Metrics& mt, const double* us, const double* vs,
                       const double* ws, const Reduce& rd, double* log, int* step, int cap) {
    // at most M blocks a plane: the partials hold M * N of each
    // (planes per block: as many as leave 2048 blocks, at most 8; whole calls with 1 plane and with the planes that
    // leave 8192, 4096, 2048 and 1024 blocks: 768 x 384 x 256 0.389, 0.336 (8 planes in all four) ms, 512 x 256 x 192
    // 0.147, 0.130, 0.131, 0.134, 0.134, 300 x 256 x 250 0.118, 0.109, 0.107, 0.108, 0.109, 300 x 128 x 256 0.072, 0.073,
    // 0.071, 0.071, 0.073, 256 x 192 x 128 0.059, 0.058, 0.059, 0.057, 0.058)
    const int nbx = std::min(span_blocks(d), d.M);
    const int planes = std::max(1, std::min(8, (int)((long)span_blocks(d) * d.N / 2048)));
    const int nb = nbx * ceil_div(d.N, planes);
    const int runs = 3 * sizeof(double) * (size_t)d.nx * d.ny * d.nz > ((size_t)256 << 20);
    hipLaunchKernelGGL(k_div_minmax, dim3(nb), dim3(256), 0, st, d, mt, us, vs, ws, rd.part, row_magic(d), nbx, planes,
                       runs);
    hipLaunchKernelGGL(k_fold_minmax, dim3(1), dim3(1024), 0, st, rd.part, nb, rd.red, log, step, cap);
}

void launch_correct(hipStream_t st, const Dims& d, const Metrics& mt, const double* us, const double* vs,
                    const double* ws, double* uo, double* vo, double* wo, const double* dp, double alfxdt,
                    int refresh_periodic, const double* dscale) {
    const CorrArgs c = corr_args(d, mt, us, vs, ws, uo, vo, wo, dp);
    const size_t cells = (size_t)d.nx * d.ny * d.nz;
    const int runs = correct_exceeds(cells, 256);
    auto go = [&](auto fn) {
        hipLaunchKernelGGL(fn, dim3(span_blocks(d) * d.N), dim3(256), 0, st, c, alfxdt, refresh_periodic, runs,
                           dscale);
    };
    if (correct_exceeds(cells, kCorrectCached)) go(k_correct_span<true>);
    else go(k_correct_span<false>);
}

void launch_laplacian(hipStream_t st, const Dims& d, const Op64& op, const double* phi, double* out) {
    hipLaunchKernelGGL(k_laplacian, cell_grid(d), kCellBlock, 0, st, d, op, phi, out);
}

void launch_finalize(hipStream_t st, const Dims& d, const Op64& op, double* phi, const double* rhs,
                     const Reduce& rd) {
    // the residual reads phi's neighbours, so it runs before the shift rewrites phi
    if (rhs) {
        hipLaunchKernelGGL(k_resid_sumsq, red_grid(d), kCellBlock, 0, st, d, op, phi, rhs, rd.part);
        launch_fold(st, rd.part, reduce_blocks(d), rd.red + RED_RNORM2);
    }
    hipLaunchKernelGGL(k_shift_ghosts, cell_grid(d), kCellBlock, 0, st, d, phi, (const double*)rd.red);
}

void launch_rhs_check(hipStream_t st, const Dims& d, const Metrics& mt, const double* b, const Reduce& rd) {
    const int nb = reduce_blocks(d);
    hipLaunchKernelGGL(k_rhs_check, red_grid(d), kCellBlock, 0, st, d, mt, b, rd.part, nb);
    launch_fold(st, rd.part, nb, rd.red + RED_CHK_VB, 3);  // RED_CHK_VB, RED_CHK_VABS, RED_CHK_NF
}

void launch_sumsq(hipStream_t st, const Dims& d, const double* a, const Reduce& rd, int slot) {
    hipLaunchKernelGGL(k_sumsq, red_grid(d), kCellBlock, 0, st, d, a, rd.part);
    launch_fold(st, rd.part, reduce_blocks(d), rd.red + slot);
}

void launch_copy_shift(hipStream_t st, const Dims& d, const double* src, double* dst, const double* red) {
    hipLaunchKernelGGL(k_copy_shift, cell_grid(d), kCellBlock, 0, st, d, src, dst, red);
}

void launch_refresh_z(hipStream_t st, const Dims& d, double* dp) {
    if (!d.cyc_z) return;
    const size_t pl = (size_t)d.nx * d.ny;
    hipLaunchKernelGGL(k_refresh_z, dim3((unsigned)((pl + 255) / 256)), dim3(256), 0, st, d, dp);
}

void launch_fill(hipStream_t st, double* p, size_t n, double v) {
    if (!n) return;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
}

}  // namespace eddy
