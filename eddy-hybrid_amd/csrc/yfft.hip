// yfft.hip -- batched real FFTs along the periodic axis (the reference's Y, 2nd index).
//
// Forward: direct.f:620-629 (RFFTF of every interior pencil DP(I+1,2:L+1,K+1));
// inverse: direct.f:1035-1106 (DUMMY/L, RFFTB, ghost fill). Output packing follows
// fftpack (fftpack.f:140-240): [Re X0, Re X1, Im X1, ..., Re X_{L/2}] (L even).
//
// Periodic lengths the radix FFT cannot take (L odd, or L/2 with a prime factor >= 7) go through
// the same tiles with the transform done as a dense real DFT on the matrix cores (the DENSE
// kernels, dft_block), the packing and scaling as above.
//
// A workgroup owns TI (a power of two) consecutive x1 pencils at one x2 index k. The pencils
// are read row by row (TI contiguous doubles per y index: coalesced), with several loads in
// flight per thread, packed as TI complex sequences z[n] = x[2n] + i x[2n+1] of length
// H = L/2 in LDS, transformed by a Stockham FFT and unpacked to the L real coefficients. The
// spectral array S keeps x1 fastest: S[i + M*(k + N*j)], so the x2 transform reads rows of
// contiguous values too.
#include <algorithm>
#include <numeric>
#include <type_traits>

#include "batch_device.h"
#include "fft_device.h"
#include "kernels.h"
#include "mma_device.h"
#include "reduce_device.h"
#include "stencil_device.h"

namespace eddy {

constexpr size_t kCacheBytes = (size_t)256 << 20;  // memory-side cache
constexpr int kLoadBatch = 8;
constexpr int kInvTasks = 2;  // packing tasks (4 coefficient rows each) per thread and load batch
constexpr int kDivRows = 4;  // rows per load sub-batch of the fused divergence and residual
// Kernel-side forms of YF_DIVERGENCE with the metric kind fixed at compile time, so that the
// Cartesian kernel does not carry the registers of the cylindrical one's divisions by RP.
constexpr int YF_DIV_CART = 3, YF_DIV_CYL = 4;

template <typename T>
struct YArgs {
    const double* src;
    const double* phi;
    const double *us, *vs, *ws;  // YF_DIVERGENCE inputs
    Metrics mt;
    double scale;
    const double* dscale;  // device {ALFXDT, 1/ALFXDT}: when non-null, scale = dscale[1]
    Op64 op;
    double* part;
    double* red;
    T* S;
    const T* Sin;
    double* dp;
    double* rhs_out;  // FP32 YF_DIVERGENCE: the FP64 divergence, DP layout
    Dims d;
    FftPlan fp;
    Tables<T> tb;
    int TI, lti;  // pencils per workgroup and its log2
    int iblk;     // forward: tiles per x1 block of the tile order (iblock_tile), 0 = whole rows
    int ld;
    int shift;
};

__device__ __forceinline__ size_t dpidx(const Dims& d, int I, int J, int K) { return sidx(d, I, J, K); }

// The metric factors of the thread's x1 index and the tile's x2 index (loaded once).
struct DivFactors {
    double cpk, apI, vx, vz, ruI, ruIm, rpI;
};

template <bool CART>
__device__ __forceinline__ DivFactors div_factors(const Metrics& mt, int gi, int k) {
    const int I = gi + 1, K = k + 1;
    DivFactors f;
    f.cpk = mt.cp[K];
    f.apI = mt.ap[I];
    f.vx = mt.volx[I];
    f.vz = mt.volz[K];
    f.ruI = CART ? 1.0 : mt.ru[I];
    f.ruIm = CART ? 1.0 : mt.ru[I - 1];
    f.rpI = CART ? 1.0 : mt.rp[I];
    return f;
}

// B cells (gi, j0 + u*jstep, k) of the forward transform's input, DIVERGENCE * scale
// (div_at's arithmetic), with sum vol*b accumulated into vsum. Every field value is loaded
// before any is used: arithmetic on a value inside the guard of its own load makes the
// compiler wait for it before the next load is issued, one load in flight per wave. Rows
// past L read row L-1 and are zeroed afterwards, as is every row when !iok.
template <int B, bool CART>
__device__ __forceinline__ void divergence_rows(const Dims& d, const Metrics& mt, const DivFactors& f,
                                                const double* __restrict__ us, const double* __restrict__ vs,
                                                const double* __restrict__ ws, double scale, int gi, bool iok,
                                                int j0, int jstep, int k, double* v, double& vsum) {
    const int I = gi + 1, K = k + 1;
    // 32-bit byte offsets from the uniform field bases (one VGPR per address; the fields are
    // far below 4 GiB): the same offset serves u, v and w
    const unsigned pl8 = 8u * (unsigned)d.nx * (unsigned)d.ny, nx8 = 8u * (unsigned)d.nx;
    double wc[B], wm[B], uc[B], um[B], vc[B], vm[B], bpJ[B], vyJ[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int J = min(j0 + u * jstep, d.L - 1) + 1;
        const unsigned o = 8u * ((unsigned)I + (unsigned)d.nx * ((unsigned)J + (unsigned)d.ny * (unsigned)K));
        wc[u] = ld_off(ws, o);
        wm[u] = ld_off(ws, o - pl8);
        uc[u] = ld_off(us, o);
        um[u] = ld_off(us, o - 8u);
        vc[u] = ld_off(vs, o);
        vm[u] = ld_off(vs, o - nx8);
    }
    // the y metric: a uniform y (DIRECT's FFT axis) takes the plan's scalars, no loads
    if (mt.bp0 != 0.0) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
            bpJ[u] = mt.bp0;
            vyJ[u] = mt.vy0;
        }
    } else {
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int J = min(j0 + u * jstep, d.L - 1) + 1;
            bpJ[u] = ld_off(mt.bp, 8u * (unsigned)J);
            vyJ[u] = ld_off(mt.voly, 8u * (unsigned)J);
        }
    }
    const double cpk = f.cpk, apI = f.apI, vx = f.vx, vz = f.vz, ruI = f.ruI, ruIm = f.ruIm, rpI = f.rpI;
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const double c = cpk * (wc[u] - wm[u]);
        double x;
        if (CART) {
            x = apI * (uc[u] - um[u]) + bpJ[u] * (vc[u] - vm[u]) + c;
        } else {
            const double ax = apI * (ruI * uc[u] - ruIm * um[u]) / rpI;
            const double bx = bpJ[u] * (vc[u] - vm[u]) / rpI;
            x = ax + bx + c;
        }
        const bool ok = iok && j0 + u * jstep < d.L;
        v[u] = ok ? x * scale : 0.0;
        vsum += ok ? vx * vyJ[u] * vz * v[u] : 0.0;  // cell_vol's product order
    }
}

// B cells of the residual r = src - L(phi) (lap_at's arithmetic); loads first, as in
// divergence_rows. The x and x2 neighbours at the walls are ghosts (in range)
// whose terms are dropped, as lap_at drops them.
template <int B>
__device__ __forceinline__ void residual_rows(const Dims& d, const Op64& op, const double* __restrict__ src,
                                              const double* __restrict__ phi, int gi, bool iok, int j0, int jstep,
                                              int k, double* v, double shift) {
    const int I = gi + 1, K = k + 1;
    // 32-bit byte offsets from the field bases (fields below 4 GiB); a neighbour step is added
    // modulo 2^32, so a negative step is its two's complement. Across a wall the neighbour is
    // the ghost (in range, its term dropped below), across a periodic x1 / x2 boundary the
    // interior cell at the other end (lap_at's coupling).
    const unsigned nx8 = 8u * (unsigned)d.nx, pl8 = nx8 * (unsigned)d.ny;
    const int i = gi;
    const unsigned oxm = (i == 0 && d.cyc_x) ? 8u * (unsigned)(d.M - 1) : 0u - 8u;
    const unsigned oxp = (i == d.M - 1 && d.cyc_x) ? 0u - 8u * (unsigned)(d.M - 1) : 8u;
    const unsigned ozm = (k == 0 && d.cyc_z) ? pl8 * (unsigned)(d.N - 1) : 0u - pl8;
    const unsigned ozp = (k == d.N - 1 && d.cyc_z) ? 0u - pl8 * (unsigned)(d.N - 1) : pl8;
    const unsigned oik = 8u * (unsigned)I + pl8 * (unsigned)K;
    double s[B], p0[B], pxm[B], pxp[B], pym[B], pyp[B], pzm[B], pzp[B];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        const int j = min(j0 + u * jstep, d.L - 1);
        const int J = j + 1;
        const int jm = (j == 0) ? d.L : J - 1;
        const int jp = (j == d.L - 1) ? 1 : J + 1;
        const unsigned o = oik + nx8 * (unsigned)J;
        s[u] = ld_off(src, o);
        p0[u] = ld_off(phi, o);
        pxm[u] = ld_off(phi, o + oxm);
        pxp[u] = ld_off(phi, o + oxp);
        pym[u] = ld_off(phi, oik + nx8 * (unsigned)jm);
        pyp[u] = ld_off(phi, oik + nx8 * (unsigned)jp);
        pzm[u] = ld_off(phi, o + ozm);
        pzp[u] = ld_off(phi, o + ozp);
    }
    const double am = op.am[i], bm = op.bm[i], cm = op.cm[i], r2 = op.r2inv[i];
    const double an = op.an[k], bn = op.bn[k], cn = op.cn[k];
    const bool xlo = i > 0 || d.cyc_x, xhi = i < d.M - 1 || d.cyc_x;
    const bool zlo = k > 0 || d.cyc_z, zhi = k < d.N - 1 || d.cyc_z;
#pragma unroll
    for (int u = 0; u < B; ++u) {
        double sx = bm * p0[u];
        if (xlo) sx += am * pxm[u];
        if (xhi) sx += cm * pxp[u];
        const double sy = (pyp[u] - 2.0 * p0[u] + pym[u]) * op.inv_delysq * r2;
        double sz = bn * p0[u];
        if (zlo) sz += an * pzm[u];
        if (zhi) sz += cn * pzp[u];
        const bool ok = iok && j0 + u * jstep < d.L;
        v[u] = ok ? (s[u] - shift) - (sx + sy + sz) : 0.0;
    }
}

// The dense real DFT of a tile, on the matrix cores. Folding the samples halves its products:
// with P_j = x_j + x_{L-j} (P_0 = x_0, P_{L/2} = x_{L/2}) and Q_j = x_j - x_{L-j} (Q_0 = 0),
//   Re X_q = sum_{j <= L/2} P_j cos(2 pi q j/L),   Im X_q = -sum_{j <= L/2} Q_j sin(2 pi q j/L),
// and the inverse takes the same two symmetric matrices over q to x_j and x_{L-j}. The plan lays
// them out in operand order (ydft_tab in api.hip: block rb of 16 outputs, step ks of 4 samples, cosine then
// sine, lane), so an operand load is one contiguous 512-byte (FP32 256-byte) read served by L2.
// A wave owns 16 outputs of 16 pencils: per step two LDS reads feed one cosine and one sine
// product, 64 matrix-core cycles each in FP64, which hide both the reads and the additions of
// the fold. L multiply-adds per value: at 160 x 96 x 112 the forward transform takes 0.029 ms and
// the inverse 0.022 ms, where a sum per output on the vector ALUs (L multiply-adds with two LDS
// reads and an index step each) took 0.716 and 0.708 ms.
constexpr int kDftAhead = 4;  // steps whose matrix operands are loaded ahead of their products

template <typename T>
struct DftAcc {
    typename Mma<T>::v4 c, s;
};

// sum over the samples of `row` (this lane's pencil) for output block rb; FOLD: the row holds x_j
// and x_{L-j} (forward), else the two operands as they are (inverse). The inverse starts from the highest
// wavenumbers: a solution's coefficients fall off with them, and a mean taken up first makes each of the
// L/2 additions after it round at its size (FP32 solves with one sweep, relative error: 20 x 6 x 254 1.07e-11
// with the mean first, 5.1e-12 last; 16 x 16 x 1001 8.2e-11 and 1.7e-11).
template <typename T, bool FOLD>
__device__ __forceinline__ DftAcc<T> dft_block(const T* __restrict__ ydm, const T* row, int nk, int rb, int lane) {
    DftAcc<T> acc;
    acc.c = typename Mma<T>::v4{T(0), T(0), T(0), T(0)};
    acc.s = acc.c;
    const T* m = ydm + (size_t)rb * nk * 128 + lane;
    const T* a = row + (lane >> 4);
    const T* b = a + 4 * nk;
    auto at = [&](int k) { return FOLD ? k : nk - 1 - k; };
    for (int k0 = 0; k0 < nk; k0 += kDftAhead) {
        T mc[kDftAhead], ms[kDftAhead];
#pragma unroll
        for (int u = 0; u < kDftAhead; ++u) {
            const int k = at(min(k0 + u, nk - 1));  // past the end: the last step's operands, unused
            mc[u] = m[k * 128];
            ms[u] = m[k * 128 + 64];
        }
#pragma unroll
        for (int u = 0; u < kDftAhead; ++u) {
            if (k0 + u < nk) {
                const T x = a[4 * at(k0 + u)], y = b[4 * at(k0 + u)];
                acc.c = Mma<T>::run(mc[u], FOLD ? x + y : x, acc.c);
                acc.s = Mma<T>::run(ms[u], FOLD ? x - y : y, acc.s);
            }
        }
    }
    return acc;
}

// Zero the slots of a tile's rows that no sample fills: 0 and the padding of both halves (and the
// second half's L/2 of an even L, its own partner).
template <typename T>
__device__ __forceinline__ void dft_zero_pads(T* rows, int pitch, int L, int TI, int tid, int nthr) {
    const int half = 4 * dft_steps(L), h = L / 2, h1 = (L - 1) / 2;
    const int na = half - 1 - h, npad = na + 1 + (half - 1 - h1);
    for (int e = tid; e < TI * npad; e += nthr) {
        const int ii = e / npad, t = e - ii * npad;
        rows[ii * pitch + (t < na ? h + 1 + t : (t == na ? half : half + h1 + t - na))] = T(0);
    }
}

// One tile (TI pencils at one x2 index) of the forward transform; `tile` is the logical tile,
// ntx the tiles per x2 row, `slot` the reduction partial's index.
template <typename T, int MODE, bool DENSE = false, bool NT = false>
__device__ __forceinline__ void yfft_fwd_tile(const YArgs<T>& a, int tile, int ntx, int slot) {
    extern __shared__ unsigned char smem_raw[];
    T* smem = reinterpret_cast<T*>(smem_raw);
    const Dims d = a.d;
    const int TI = a.TI, lti = a.lti, ld = a.ld, H = d.L / 2, L = d.L;
    // FFT: TI complex rows (split re/im) transformed in place, then the two twiddle tables;
    // DENSE: TI real rows, x_j (j <= L/2) at j and x_{L-j} at 4 dft_steps(L) + j
    T* Ar = smem;
    T* Ai = Ar + TI * ld;
    T* twc_r = Ai + TI * ld;  // exp(-2 pi i t/H), t < H
    T* twc_i = twc_r + H;
    T* twr_r = twc_i + H;  // exp(-2 pi i k/L), k <= H
    T* twr_i = twr_r + H + 1;
    const int i0 = (tile % ntx) * TI;
    const int k = tile / ntx;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int total = TI * L;
    if (DENSE) {
        dft_zero_pads<T>(Ar, ld, L, TI, tid, nthr);
    } else {
        for (int t = tid; t <= H; t += nthr) {
            if (t < H) {
                twc_r[t] = a.tb.ytwc_re[t];
                twc_i[t] = a.tb.ytwc_im[t];
            }
            twr_r[t] = a.tb.ytwr_re[t];
            twr_i[t] = a.tb.ytwr_im[t];
        }
    }

    double shift = 0.0;
    if ((MODE == YF_DIRECT || MODE == YF_RESIDUAL) && a.shift) shift = a.red[RED_VOLB] / a.red[RED_VOL];
    double rsq = 0.0;
    // The thread's x1 offset is fixed (blockDim is a multiple of TI); its rows are
    // j0, j0 + jstep, ... Rows past L and pencils past M read a clamped in-range cell and are
    // zeroed after the loads, so each batch issues all its loads before using any.
    const int ii = tid & (TI - 1);
    const bool iok = i0 + ii < d.M;
    const int gi = iok ? i0 + ii : d.M - 1;
    const int jstep = nthr >> lti;
    auto put = [&](double x, int j) {  // row j of pencil ii into the packed complex buffer
        if (j < L) {
            if (DENSE) Ar[ii * ld + (j <= H ? j : 4 * dft_steps(L) + L - j)] = T(x);
            else if (j & 1) Ai[ii * ld + pidx((j >> 1))] = T(x);
            else Ar[ii * ld + pidx((j >> 1))] = T(x);
        }
    };
    for (int e0 = tid; e0 < total; e0 += nthr * kLoadBatch) {
        const int j0 = e0 >> lti;
        if (MODE == YF_DIRECT) {
            // 32-bit byte offsets from the field base (DP < 4 GiB)
            const unsigned nx8 = 8u * (unsigned)d.nx;
            const unsigned ok0 = nx8 * (unsigned)d.ny * (unsigned)(k + 1) + 8u * (unsigned)(gi + 1);
            double x[kLoadBatch];
#pragma unroll
            for (int u = 0; u < kLoadBatch; ++u) {
                const int j = min(j0 + u * jstep, L - 1);
                x[u] = ld_off(a.src, ok0 + nx8 * (unsigned)(j + 1));
            }
#pragma unroll
            for (int u = 0; u < kLoadBatch; ++u) put((iok && j0 + u * jstep < L) ? x[u] - shift : 0.0, j0 + u * jstep);
        } else if (MODE == YF_RESIDUAL) {
#pragma unroll
            for (int h = 0; h < kLoadBatch / kDivRows; ++h) {  // sub-batches as for the divergence below
                const int jh = j0 + h * kDivRows * jstep;
                double v[kDivRows];
                residual_rows<kDivRows>(d, a.op, a.src, a.phi, gi, iok, jh, jstep, k, v, shift);
#pragma unroll
                for (int r = 0; r < kDivRows; ++r) put(v[r], jh + r * jstep);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            const bool cart = MODE == YF_DIV_CART || (MODE == YF_DIVERGENCE && a.mt.cart);
            const DivFactors f = cart ? div_factors<true>(a.mt, gi, k) : div_factors<false>(a.mt, gi, k);
            const double scale = a.dscale ? a.dscale[1] : a.scale;
            // sub-batches of kDivRows rows: the loads of one sub-batch are in flight together;
            // the scheduling barrier keeps the compiler from hoisting the next sub-batch's loads
            // above this one's arithmetic, which would need registers for all of them at once
#pragma unroll
            for (int h = 0; h < kLoadBatch / kDivRows; ++h) {
                const int jh = j0 + h * kDivRows * jstep;
                double v[kDivRows];
                if (cart)
                    divergence_rows<kDivRows, true>(d, a.mt, f, a.us, a.vs, a.ws, scale, gi, iok, jh, jstep, k, v,
                                                    rsq);
                else
                    divergence_rows<kDivRows, false>(d, a.mt, f, a.us, a.vs, a.ws, scale, gi, iok, jh, jstep, k, v,
                                                     rsq);
#pragma unroll
                for (int r = 0; r < kDivRows; ++r) put(v[r], jh + r * jstep);
                if constexpr (std::is_same<T, float>::value) {
                    // the FP64 RHS of the defect correction, stored beside the FP32 transform
                    // input (the refined projection forms it nowhere else)
                    if (iok && a.rhs_out) {
                        const unsigned nx8 = 8u * (unsigned)d.nx;
                        const unsigned ok0 = nx8 * (unsigned)d.ny * (unsigned)(k + 1) + 8u * (unsigned)(gi + 1);
#pragma unroll
                        for (int r = 0; r < kDivRows; ++r)
                            if (jh + r * jstep < L) st_off(a.rhs_out, ok0 + nx8 * (unsigned)(jh + r * jstep + 1), v[r]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    if (MODE == YF_DIVERGENCE || MODE == YF_DIV_CART || MODE == YF_DIV_CYL)
        block_partial<RED_OP_SUM>(rsq, a.part, slot);
    __syncthreads();
    const size_t js = (size_t)d.M * (size_t)d.N;
    T* outK = a.S + (size_t)d.M * (size_t)k;
    if (DENSE) {
        // item: 16 wavenumbers of 16 pencils to a wave (fewer pencils in the tile: the lanes past
        // TI repeat a row and store nothing); packed slots 2q-1 (Re) and 2q (Im), slot 0 Re X_0
        const int nk = dft_steps(L), nrb = dft_blocks(L), ncb = (TI + 15) >> 4;
        const int lane = tid & 63;
        for (int it = __builtin_amdgcn_readfirstlane(tid >> 6); it < nrb * ncb; it += nthr >> 6) {
            const int rb = it / ncb, p = 16 * (it - rb * ncb) + (lane & 15);
            const DftAcc<T> r = dft_block<T, true>(a.tb.ydm, Ar + (p & (TI - 1)) * ld, nk, rb, lane);
            const int gi = i0 + p;
            if (p >= TI || gi >= d.M) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = 16 * rb + Mma<T>::row(lane >> 4, v);
                if (q <= H) outK[js * (size_t)(q ? 2 * q - 1 : 0) + gi] = r.c[v];
                if (q > 0 && 2 * q < L) outK[js * (size_t)(2 * q) + gi] = -r.s[v];
            }
        }
        return;
    }
    if (H > 1) cfft_lds<T>(Ar, Ai, ld, TI, a.fp, twc_r, twc_i, T(-1), tid, nthr);
    const T* Zr = Ar;
    const T* Zi = Ai;
    // X_k = (Z_k + conj Z_{H-k})/2 - i W^k (Z_k - conj Z_{H-k})/2, W = exp(-2 pi i/L). The
    // thread's pencil is fixed (blockDim is a multiple of TI); its coefficients k step by
    // blockDim/TI. S addresses as 32-bit byte offsets from the tile's column (S < 4 GiB).
    {
        const int ii = tid & (TI - 1);
        const int gi = i0 + ii;
        if (gi < d.M) {
            const T* zr = Zr + ii * ld;
            const T* zi = Zi + ii * ld;
            T* out = outK + gi;
            const unsigned jsb = (unsigned)(js * sizeof(T));
            const int kstep = nthr >> lti;
            for (int kk = tid >> lti; kk <= H; kk += kstep) {
                const int k1 = (kk == H) ? 0 : kk;
                const int k2 = (kk == 0) ? 0 : H - kk;
                const T ar = zr[pidx(k1)], ai = zi[pidx(k1)];
                const T br = zr[pidx(k2)], bi = -zi[pidx(k2)];
                const T er = T(0.5) * (ar + br), ei = T(0.5) * (ai + bi);
                const T dr = T(0.5) * (ar - br), di = T(0.5) * (ai - bi);
                const T wr = twr_r[kk], wi = twr_i[kk];
                const T wdr = wr * dr - wi * di, wdi = wr * di + wi * dr;
                const T xr = er + wdi, xi = ei - wdr;
                if (kk == 0) {
                    st_once<NT>(out, 0u, xr);
                } else if (kk == H) {
                    st_once<NT>(out, jsb * (unsigned)(L - 1), xr);
                } else {
                    st_once<NT>(out, jsb * (unsigned)(2 * kk - 1), xr);
                    st_once<NT>(out, jsb * (unsigned)(2 * kk), xi);
                }
            }
        }
    }
}

// NT: the spectrum's rows are whole lines (M a multiple of 16) and it fills the 256 MiB memory-side
// cache, which non-temporal stores leave to the velocities (512 x 256 x 256: this kernel 0.2746 -> 0.2727 ms,
// the line solve 0.1148 -> 0.1097). Rows that begin inside a line lose by it (500 x 256 x 256 0.278 -> 0.327),
// and smaller spectra are read back from the cache (256 x 192 x 128: x2 transform 0.0284 -> 0.0320). Whole
// projections without and with it, by the size of the spectrum: 72 MiB 0.3170 -> 0.3210 ms and 0.3274 -> 0.3310; 112 and
// 117 equal; 160 0.6912 -> 0.6910; 192 0.8005 -> 0.7976, 0.8083 -> 0.8052 and 0.7728 -> 0.7784; 240 0.9968 -> 0.9965;
// 256 1.0620 -> 1.0509 and 1.0678 -> 1.0591; 288 1.2742 -> 1.2685; 320 1.4172 -> 1.4092; 384 to 960 within 0.4 % of each
// other, both ways. Solves of a stored RHS: 256 0.5616 -> 0.5604, 288 0.7231 -> 0.7216, 320 0.7908 -> 0.7960, 384
// 0.9014 -> 0.9094, 480 1.1504 -> 1.1566, 960 2.4089 -> 2.4001.
template <typename T, int MODE, bool DENSE, bool NT = false>
__global__ void __launch_bounds__(kFftThreads) k_yfft_fwd(YArgs<T> a) {
    const int nb = gridDim.x * gridDim.y;
    const int t = iblock_tile(xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, nb), gridDim.x, gridDim.y, a.iblk);
    yfft_fwd_tile<T, MODE, DENSE, NT>(a, t, gridDim.x, linear_bid());
}

// The forward transform of a stored RHS at no more than 80 VGPRs: with its 42 KB LDS tile
// (L = 256, 16 pencils) three workgroups of 8 waves then share a CU (6 waves per SIMD).
template <typename T, bool DENSE, bool NT = false>
__global__ void __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(6))) k_yfft_fwd_rhs(YArgs<T> a) {
    const int nb = gridDim.x * gridDim.y;
    const int t = iblock_tile(xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, nb), gridDim.x, gridDim.y, a.iblk);
    yfft_fwd_tile<T, YF_DIRECT, DENSE, NT>(a, t, gridDim.x, linear_bid());
}

template <typename T, int MODE, bool DENSE = false, bool NT = false>
__device__ __forceinline__ void yfft_inv_tile(const YArgs<T>& a, int tile, int ntx, int slot) {
    extern __shared__ unsigned char smem_raw[];
    T* smem = reinterpret_cast<T*>(smem_raw);
    const Dims d = a.d;
    const int TI = a.TI, lti = a.lti, ld = a.ld, H = d.L / 2, L = d.L;
    T* Ar = smem;  // FFT: TI complex rows, transformed in place; DENSE: TI rows of coefficients
    T* Ai = Ar + TI * ld;
    T* twc_r = Ai + TI * ld;
    T* twc_i = twc_r + H;
    T* twr_r = twc_i + H;
    T* twr_i = twr_r + H + 1;
    const int i0 = (tile % ntx) * TI;
    const int k = tile / ntx;
    const int tid = threadIdx.x, nthr = blockDim.x;
    if (DENSE) {
        dft_zero_pads<T>(Ar, ld, L, TI, tid, nthr);
    } else {
        for (int t = tid; t <= H; t += nthr) {
            if (t < H) {
                twc_r[t] = a.tb.ytwc_re[t];
                twc_i[t] = a.tb.ytwc_im[t];
            }
            twr_r[t] = a.tb.ytwr_re[t];
            twr_i[t] = a.tb.ytwr_im[t];
        }
    }
    const size_t js = (size_t)d.M * (size_t)d.N;
    const T* inK = a.Sin + (size_t)d.M * (size_t)k;
    __syncthreads();  // the twiddle tables are read below by other threads than wrote them
    if (DENSE) {
        // the packed coefficients of the tile's pencils into LDS rows (rows of contiguous x1
        // values: coalesced): w_q Re X_q / L at q and -2 Im X_q / L at 4 dft_steps(L) + q, with
        // w = 1 for q = 0 and L/2 (their own partners), else 2; pencils past M read a clamped row
        const T invL = T(1) / T(L), inv2 = T(2) * invL;
        const int ii = tid & (TI - 1), half = 4 * dft_steps(L);
        const bool iok = i0 + ii < d.M;
        const T* col = inK + (iok ? i0 + ii : d.M - 1);
        const int sstep = nthr >> lti;
        for (int s0 = tid >> lti; s0 < L; s0 += sstep * kLoadBatch) {
            T x[kLoadBatch];
#pragma unroll
            for (int u = 0; u < kLoadBatch; ++u) x[u] = col[js * (size_t)min(s0 + u * sstep, L - 1)];
#pragma unroll
            for (int u = 0; u < kLoadBatch; ++u) {
                const int s = s0 + u * sstep, q = (s + 1) >> 1;
                const bool re = s == 0 || (s & 1);
                const T w = !iok ? T(0) : (!re ? -inv2 : ((q == 0 || 2 * q == L) ? invL : inv2));
                if (s < L) Ar[ii * ld + (re ? q : half + q)] = iok ? x[u] * w : T(0);
            }
        }
        __syncthreads();
    }

    // Packed spectrum -> Z'_q = [(X_q + conj X_{H-q}) + i conj(W^q) (X_q - conj X_{H-q})] / L,
    // q < H. Task (ii, q) for q <= H/2 reads the coefficient rows of X_q and X_{H-q} straight
    // from S (X_0 = row 0, X_H = row L-1, X_p = rows 2p-1, 2p otherwise) and forms Z'_q and
    // Z'_{H-q}: every row is read once and nothing is staged.
    const T invL = T(1) / T(L);
    const int half = DENSE ? -1 : H / 2;  // DENSE: no packing tasks
    constexpr int UB = kInvTasks;
    // The thread's x1 offset is fixed (blockDim is a multiple of TI). The four coefficient
    // rows of a task are loaded before any arithmetic (arithmetic inside a load's own guard
    // makes the compiler wait for it before the next load): rows 2q-1, 2q, 2(H-q)-1, 2(H-q),
    // with q = 0 reading rows 0 and L-1 (X_0, X_H real). Tasks past H/2 and pencils past M
    // read clamped in-range rows whose values are zeroed afterwards.
    const int ii = tid & (TI - 1);
    const bool iok = i0 + ii < d.M;
    const T* col = inK + (iok ? i0 + ii : d.M - 1);
    const int qstep = nthr >> lti;
    // Row addresses as 32-bit byte offsets from the column (S < 4 GiB), stepped with the task
    // index instead of multiplied: with rs the bytes between coefficient rows and
    // qo = 2 q rs, rows 2q-1, 2q, 2(H-q)-1 and 2(H-q) are qo - rs, qo, (L-1) rs - qo and
    // L rs - qo (q = 0: rows 0, 1, L-1 and L-1 again). Tasks past H/2 take task H/2's rows.
    const unsigned rs = (unsigned)sizeof(T) * (unsigned)d.M * (unsigned)d.N;
    const unsigned lm1 = (unsigned)(L - 1) * rs;
    const unsigned q2 = 2u * rs, qcap = (unsigned)half * q2;
    unsigned qo0 = (unsigned)(tid >> lti) * q2;
    for (int q0 = tid >> lti; q0 <= half; q0 += qstep * UB, qo0 += (unsigned)(qstep * UB) * q2) {
        T xa_r[UB], xa_i[UB], xb_r[UB], xb_i[UB];
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const unsigned qo = (q0 + u * qstep <= half) ? qo0 + (unsigned)(u * qstep) * q2 : qcap;
            const bool q0row = qo == 0;
            const unsigned ob = lm1 - qo;
            xa_r[u] = ld_once<NT>(col, q0row ? 0u : qo - rs);
            xa_i[u] = ld_once<NT>(col, q0row ? rs : qo);
            xb_r[u] = ld_once<NT>(col, ob);
            xb_i[u] = ld_once<NT>(col, q0row ? lm1 : ob + rs);
        }
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const int q = q0 + u * qstep;
            if (q > half) continue;
            const bool im = iok && q > 0;
            xa_r[u] = iok ? xa_r[u] : T(0);
            xb_r[u] = iok ? xb_r[u] : T(0);
            xa_i[u] = im ? xa_i[u] : T(0);
            xb_i[u] = im ? xb_i[u] : T(0);
            const int qb = H - q;
            T* rr = Ar + ii * ld;
            T* ri = Ai + ii * ld;
            {
                const T yr = xb_r[u], yi = -xb_i[u];
                const T sr = xa_r[u] + yr, si = xa_i[u] + yi;
                const T dr = xa_r[u] - yr, di = xa_i[u] - yi;
                const T wr = twr_r[q], wi = -twr_i[q];
                const T vr = wr * dr - wi * di, vi = wr * di + wi * dr;
                rr[pidx(q)] = (sr - vi) * invL;
                ri[pidx(q)] = (si + vr) * invL;
            }
            if (qb < H && qb != q) {
                const T yr = xa_r[u], yi = -xa_i[u];
                const T sr = xb_r[u] + yr, si = xb_i[u] + yi;
                const T dr = xb_r[u] - yr, di = xb_i[u] - yi;
                const T wr = twr_r[qb], wi = -twr_i[qb];
                const T vr = wr * dr - wi * di, vi = wr * di + wi * dr;
                rr[pidx(qb)] = (sr - vi) * invL;
                ri[pidx(qb)] = (si + vr) * invL;
            }
        }
    }
    if (!DENSE) {
        __syncthreads();
        if (H > 1) cfft_lds<T>(Ar, Ai, ld, TI, a.fp, twc_r, twc_i, T(1), tid, nthr);
    }
    const T* Zr = Ar;
    const T* Zi = Ai;
    double psum = 0.0;
    const int K = k + 1;
    const double mean =
        MODE == YI_UPDATE_FINAL ? a.red[RED_PHISUM] / ((double)d.M * (double)d.L * (double)d.N) : 0.0;
    const int total = TI * L;
    // DP addresses as 32-bit byte offsets from the field base (DP < 4 GiB)
    const unsigned nx8 = 8u * (unsigned)d.nx, pl8K = nx8 * (unsigned)d.ny * (unsigned)K;
    // the value v of cell (gi, j) of the plane, as MODE stores it
    auto emit = [&](int gi, int j, double v) {
        const unsigned oj = pl8K + nx8 * (unsigned)(j + 1) + 8u * (unsigned)(gi + 1);
        const int I = gi + 1, J = j + 1;
        if (MODE == YI_UPDATE_FINAL) v = ld_off(a.dp, oj) + v - mean;
        if (MODE == YI_DIRECT || MODE == YI_UPDATE_FINAL) {
            // interior plus the x ghosts (MP=1: DP(1)=DP(2), DP(NX)=DP(NX-1); MP=0: DP(1)=DP(NX-1),
            // DP(NX)=DP(2)) and the y ghosts (LP=0: DP(:,1)=DP(:,NY-1), DP(:,NY)=DP(:,2); LP=1:
            // DP(:,1)=DP(:,2), DP(:,NY)=DP(:,NY-1)), direct.f:1090-1106
            st_off(a.dp, oj, v);
            const int Ilo = (gi == (d.cyc_x ? d.M - 1 : 0)) ? 0 : -1;
            const int Ihi = (gi == (d.cyc_x ? 0 : d.M - 1)) ? d.nx - 1 : -1;
            const int Jg = d.ycopy ? ((j == 0) ? 0 : ((j == L - 1) ? d.ny - 1 : -1))
                                   : ((j == L - 1) ? 0 : ((j == 0) ? d.ny - 1 : -1));
            if (Ilo >= 0) a.dp[dpidx(d, Ilo, J, K)] = v;
            if (Ihi >= 0) a.dp[dpidx(d, Ihi, J, K)] = v;
            if (Jg >= 0) {
                a.dp[dpidx(d, I, Jg, K)] = v;
                if (Ilo >= 0) a.dp[dpidx(d, Ilo, Jg, K)] = v;
                if (Ihi >= 0) a.dp[dpidx(d, Ihi, Jg, K)] = v;
            }
        } else if (MODE == YI_STORE) {
            st_off(a.dp, oj, v);
            psum += v;
        } else {
            const double nv = ld_off(a.dp, oj) + v;
            st_off(a.dp, oj, nv);
            psum += nv;
        }
    };
    if (DENSE) {
        // x_j = E_j + O_j and x_{L-j} = E_j - O_j, E and O the cosine and sine sums (fftpack's
        // RFFTB after direct.f:1036)
        const int nk = dft_steps(L), nrb = dft_blocks(L), ncb = (TI + 15) >> 4;
        const int lane = tid & 63;
        for (int it = __builtin_amdgcn_readfirstlane(tid >> 6); it < nrb * ncb; it += nthr >> 6) {
            const int rb = it / ncb, p = 16 * (it - rb * ncb) + (lane & 15);
            const DftAcc<T> r = dft_block<T, false>(a.tb.ydm, Ar + (p & (TI - 1)) * ld, nk, rb, lane);
            const int gi = i0 + p;
            if (p >= TI || gi >= d.M) continue;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int j = 16 * rb + Mma<T>::row(lane >> 4, v);
                if (j <= H) emit(gi, j, (double)(r.c[v] + r.s[v]));
                if (j > 0 && 2 * j < L) emit(gi, L - j, (double)(r.c[v] - r.s[v]));
            }
        }
    } else {
        for (int e = tid; e < total; e += nthr) {
            const int ii = e & (TI - 1);
            const int j = e >> lti;
            if (i0 + ii >= d.M) continue;
            emit(i0 + ii, j, (double)((j & 1) ? Zi[ii * ld + pidx((j >> 1))] : Zr[ii * ld + pidx((j >> 1))]));
        }
    }
    if (MODE == YI_DIRECT || MODE == YI_UPDATE_FINAL) {
        // z ghost planes (K=1, K=NZ) are zero (direct.f:1035); the blocks at the two ends
        // of x2 clear them for their x1 range (with the x ghosts at the domain edges).
        if (k == 0 || k == d.N - 1) {
            const int Kg = (k == 0) ? 0 : d.nz - 1;
            const int ilo = (i0 == 0) ? 0 : i0 + 1;
            const int ihi = (i0 + TI >= d.M) ? d.nx - 1 : i0 + TI;
            const int w = ihi - ilo + 1;
            for (int e = tid; e < w * d.ny; e += nthr) {
                const int I = ilo + e % w;
                const int J = e / w;
                a.dp[dpidx(d, I, J, Kg)] = 0.0;
            }
        }
    } else {
        block_partial<RED_OP_SUM>(psum, a.part, slot);
    }
}

// NT: the spectrum's rows are whole lines and it fills the memory-side cache with the pressure; its
// last read, past the caches, leaves them the pressure for CORRECT (512 x 256 x 256: this kernel 0.137 -> 0.131 ms
// and CORRECT 0.343 -> 0.330; 512 x 256 x 192 0.100 -> 0.089 and 0.256 -> 0.244; 768 x 384 x 256 0.278 -> 0.259 but
// CORRECT 0.777 -> 0.795). Whole projections without and with it: spectra of 117 MiB 0.5578 -> 0.5567 ms, 128 0.5243 ->
// 0.5162, 160 0.7037 -> 0.6912, 192 0.8237 -> 0.8005, 256 1.0771 -> 1.0620, 320 1.4175 -> 1.4172; past that within 0.7 % of
// each other, both ways (768 x 384 x 256 2.4607 -> 2.4603). A smaller spectrum (72 MiB 0.3281 -> 0.3338) comes from the caches, and lines that two tiles share would be
// read twice (300 x 256 x 250: 0.084 -> 0.097 and 0.195 -> 0.187; 300 x 128 x 128 0.0252 -> 0.0280).
template <typename T, int MODE, bool DENSE, bool NT = false>
// at most 80 VGPRs (the last defect-correction update needs 82 unbounded): with its 42 KB LDS
// tile (L = 256, 16 pencils) three workgroups of 8 waves share a CU (6 waves per SIMD)
__global__ void __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(6))) k_yfft_inv(YArgs<T> a) {
    yfft_inv_tile<T, MODE, DENSE, NT>(a, xcd_tile(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y), gridDim.x,
                                  linear_bid());
}

// TI complex rows (transformed in place) + the two twiddle tables
static inline size_t ylds_bytes(int TI, int ld, size_t tsz) { return (2 * (size_t)TI * ld + 4 * (size_t)ld) * tsz; }
// the dense DFT: TI real rows
static inline size_t ylds_dense_bytes(int TI, int L, size_t tsz) { return (size_t)TI * dft_pitch(L) * tsz; }

static inline int ilog2(int v) {
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

template <typename T>
void launch_yfft_fwd(hipStream_t st, const Dims& d, const FftPlan& fp, const Tables<T>& tb, const FwdInput& in,
                     const Op64& op, const Reduce& rd, T* S, int TI, int iblk) {
    if constexpr (std::is_same<T, float>::value) {
        if (tb.ydft_f && (in.mode == YF_DIRECT || in.mode == YF_RESIDUAL)) {
            launch_ygemm_fwd(st, d, tb.ydft_f, in, op, rd, S);
            return;
        }
    }
    const double* src = in.src;
    const double* phi = in.phi;
    const int shift = in.shift;
    const int mode = in.mode;
    YArgs<T> a{};
    a.src = src;
    a.phi = phi;
    a.rhs_out = in.rhs_out;
    a.op = op;
    a.part = rd.part;
    a.red = rd.red;
    a.S = S;
    a.d = d;
    a.fp = fp;
    a.tb = tb;
    a.TI = TI;
    a.lti = ilog2(TI);
    a.iblk = iblk;
    const bool dense = fp.n == 0;  // the plan's dense-DFT marker (no radix plan for L)
    a.ld = dense ? dft_pitch(d.L) : fft_ld(d.L / 2);
    a.shift = shift;
    dim3 grid(ceil_div(d.M, TI), d.N);
    size_t sh = dense ? ylds_dense_bytes(TI, d.L, sizeof(T)) : ylds_bytes(TI, a.ld, sizeof(T));
    auto go = [&](auto fn) {
        (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
        hipLaunchKernelGGL(fn, grid, dim3(kFftThreads), sh, st, a);
    };
    constexpr bool F64 = std::is_same<T, double>::value;
    const size_t spectrum = sizeof(T) * (size_t)d.M * d.N * d.L;
    const bool once = F64 && d.M % 16 == 0 && spectrum >= kCacheBytes;
    if (mode == YF_DIRECT) {
        if (dense) go(k_yfft_fwd<T, YF_DIRECT, true>);
        else if (once) go(k_yfft_fwd_rhs<T, false, F64>);
        else go(k_yfft_fwd_rhs<T, false>);
    } else if (mode == YF_DIVERGENCE) {
        a.us = in.us;
        a.vs = in.vs;
        a.ws = in.ws;
        a.mt = in.mt;
        a.scale = in.scale;
        a.dscale = in.dscale;
        if (dense) {
            if (in.mt.cart) go(k_yfft_fwd<T, YF_DIV_CART, true>);
            else go(k_yfft_fwd<T, YF_DIV_CYL, true>);
        } else {
            if (in.mt.cart && once) go(k_yfft_fwd<T, YF_DIV_CART, false, F64>);
            else if (in.mt.cart) go(k_yfft_fwd<T, YF_DIV_CART, false>);
            else if (once) go(k_yfft_fwd<T, YF_DIV_CYL, false, F64>);
            else go(k_yfft_fwd<T, YF_DIV_CYL, false>);
        }
        if (in.fold) {
            launch_fold(st, rd.part, (int)(grid.x * grid.y), rd.red + RED_VOLB, 1, in.mt.vol_total);
        }
    } else {
        if (dense) go(k_yfft_fwd<T, YF_RESIDUAL, true>);
        else go(k_yfft_fwd<T, YF_RESIDUAL, false>);
    }
}

template <typename T>
void launch_yfft_inv(hipStream_t st, const Dims& d, const FftPlan& fp, const Tables<T>& tb,
                     const T* S, double* dp, const Reduce& rd, int TI, int mode, bool fold) {
    if constexpr (std::is_same<T, float>::value) {
        if (tb.ydft_b && (mode == YI_STORE || mode == YI_UPDATE)) {
            launch_ygemm_inv(st, d, tb.ydft_b, S, dp, rd, mode, fold);
            return;
        }
    }
    YArgs<T> a{};
    a.Sin = S;
    a.dp = dp;
    a.part = rd.part;
    a.red = rd.red;
    a.d = d;
    a.fp = fp;
    a.tb = tb;
    a.TI = TI;
    a.lti = ilog2(TI);
    const bool dense = fp.n == 0;
    a.ld = dense ? dft_pitch(d.L) : fft_ld(d.L / 2);
    dim3 grid(ceil_div(d.M, TI), d.N);
    size_t sh = dense ? ylds_dense_bytes(TI, d.L, sizeof(T)) : ylds_bytes(TI, a.ld, sizeof(T));
    auto go = [&](auto fn) {
        (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
        hipLaunchKernelGGL(fn, grid, dim3(kFftThreads), sh, st, a);
    };
    constexpr bool F64 = std::is_same<T, double>::value;
    const size_t spectrum = sizeof(T) * (size_t)d.M * d.N * d.L;
    switch (mode) {
        case YI_DIRECT:
            if (dense) go(k_yfft_inv<T, YI_DIRECT, true>);
            else if (F64 && d.M % 16 == 0 && 2 * spectrum >= kCacheBytes) go(k_yfft_inv<T, YI_DIRECT, false, F64>);
            else go(k_yfft_inv<T, YI_DIRECT, false>);
            break;
        case YI_STORE:
            if (dense) go(k_yfft_inv<T, YI_STORE, true>);
            else go(k_yfft_inv<T, YI_STORE, false>);
            if (fold) launch_fold(st, rd.part, (int)(grid.x * grid.y), rd.red + RED_PHISUM);
            break;
        case YI_UPDATE_FINAL:
            if (dense) go(k_yfft_inv<T, YI_UPDATE_FINAL, true>);
            else go(k_yfft_inv<T, YI_UPDATE_FINAL, false>);
            break;
        default:
            if (dense) go(k_yfft_inv<T, YI_UPDATE, true>);
            else go(k_yfft_inv<T, YI_UPDATE, false>);
            if (fold) launch_fold(st, rd.part, (int)(grid.x * grid.y), rd.red + RED_PHISUM);
            break;
    }
}

// ------------------------------------------------------------------ batched (one item per workgroup)
// The residual form at no more than 128 VGPRs (129 unbounded): two workgroups of 8 waves per
// CU instead of one, as its plan kernel runs.
template <typename T, int MODE>
__global__ void __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(MODE == YF_RESIDUAL ? 4 : 1)))
k_batch_yfft_fwd(const Job<YArgs<T>>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total,
             [](const Job<YArgs<T>>& J, int t) { yfft_fwd_tile<T, MODE>(J.a, t, J.ntx, t); });
}

// the stored-RHS form at no more than 80 VGPRs, as k_yfft_fwd_rhs
template <typename T>
__global__ void __launch_bounds__(kFftThreads) __attribute__((amdgpu_waves_per_eu(6)))
k_batch_yfft_fwd_rhs(const Job<YArgs<T>>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total,
             [](const Job<YArgs<T>>& J, int t) { yfft_fwd_tile<T, YF_DIRECT>(J.a, t, J.ntx, t); });
}

template <typename T, int MODE>
__global__ void __launch_bounds__(kFftThreads) k_batch_yfft_inv(const Job<YArgs<T>>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total, [](const Job<YArgs<T>>& J, int t) { yfft_inv_tile<T, MODE>(J.a, t, J.ntx, t); });
}

template <typename T>
static YArgs<T> yargs_of(const BatchProblem<T>& p, int fwd, int mode) {
    YArgs<T> a{};
    a.d = p.d;
    a.fp = p.fpy;
    a.tb = p.tb;
    a.TI = p.tiy;
    a.lti = ilog2(p.tiy);
    a.ld = fft_ld(p.d.L / 2);
    a.part = p.part;
    a.red = p.red;
    a.op = p.op;
    if (fwd) {
        a.S = p.S;
        if (mode == YF_DIRECT) {
            a.src = p.rhs ? p.rhs : p.dp;
        } else if (mode == YF_RESIDUAL) {
            a.src = p.rhs;
            a.phi = p.dp;
        } else {
            a.us = p.us;
            a.vs = p.vs;
            a.ws = p.ws;
            a.mt = p.mt;
            a.dscale = p.dscale;
        }
    } else {
        a.Sin = p.S;
        a.dp = p.dp;
    }
    return a;
}


template <typename T>
int prepare_yfft(const std::vector<BatchProblem<T>>& pr, int fwd, int mode, StageLaunch& out,
                 std::vector<void*>& owned) {
    auto lds_of = [&](int x) { return ylds_bytes(pr[x].tiy, fft_ld(pr[x].d.L / 2), sizeof(T)); };
    std::vector<int> order(pr.size());
    std::iota(order.begin(), order.end(), 0);
    // the tiles of most LDS (fewest workgroups per CU) first, then the longest
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
        const int ox = lds_occupancy(lds_of(x)), oy = lds_occupancy(lds_of(y));
        return ox != oy ? ox < oy : pr[x].tiy * pr[x].d.L > pr[y].tiy * pr[y].d.L;
    });
    std::vector<Job<YArgs<T>>> jobs;
    out = StageLaunch{};
    for (int idx : order) {
        const BatchProblem<T>& p = pr[idx];
        Job<YArgs<T>> j{};
        j.a = yargs_of(p, fwd, mode);
        j.ntx = ceil_div(p.d.M, p.tiy);
        j.ntiles = j.ntx * p.d.N;
        if (!add_class_job(out, jobs, j, 0, lds_of(idx))) return -1;
    }
    if (upload_jobs(jobs, out, owned)) return -1;
    if (fwd && mode == YF_DIVERGENCE && !pr.empty()) {
        bool all_cart = true, all_cyl = true;
        for (const BatchProblem<T>& p : pr) {
            all_cart = all_cart && p.mt.cart;
            all_cyl = all_cyl && !p.mt.cart;
        }
        out.kind = all_cart ? 1 : (all_cyl ? 2 : 0);
    }
    return 0;
}

template <typename T>
void batch_yfft(hipStream_t st, const StageLaunch& sl, int fwd, int mode) {
    auto go = [&](auto fn) {
        (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sl.lds);
        for (int c = 0; c < sl.ncls; ++c) {
            const Job<YArgs<T>>* jobs = (const Job<YArgs<T>>*)sl.jobs + sl.cls_job[c];
            hipLaunchKernelGGL(fn, dim3(std::max(sl.cls_total[c], 1)), dim3(kFftThreads), sl.cls_lds[c], st, jobs,
                               sl.cls_job[c + 1] - sl.cls_job[c], sl.cls_total[c]);
        }
    };
    if (fwd) {
        if (mode == YF_DIRECT) go(k_batch_yfft_fwd_rhs<T>);
        else if (mode == YF_RESIDUAL) go(k_batch_yfft_fwd<T, YF_RESIDUAL>);
        else if (sl.kind == 1) go(k_batch_yfft_fwd<T, YF_DIV_CART>);
        else if (sl.kind == 2) go(k_batch_yfft_fwd<T, YF_DIV_CYL>);
        else go(k_batch_yfft_fwd<T, YF_DIVERGENCE>);
    } else {
        if (mode == YI_DIRECT) go(k_batch_yfft_inv<T, YI_DIRECT>);
        else if (mode == YI_STORE) go(k_batch_yfft_inv<T, YI_STORE>);
        else go(k_batch_yfft_inv<T, YI_UPDATE>);
    }
}

template int prepare_yfft<double>(const std::vector<BatchProblem<double>>&, int, int, StageLaunch&,
                                  std::vector<void*>&);
template int prepare_yfft<float>(const std::vector<BatchProblem<float>>&, int, int, StageLaunch&,
                                 std::vector<void*>&);
template void batch_yfft<double>(hipStream_t, const StageLaunch&, int, int);
template void batch_yfft<float>(hipStream_t, const StageLaunch&, int, int);

template void launch_yfft_fwd<double>(hipStream_t, const Dims&, const FftPlan&, const Tables<double>&,
                                      const FwdInput&, const Op64&, const Reduce&, double*, int, int);
template void launch_yfft_fwd<float>(hipStream_t, const Dims&, const FftPlan&, const Tables<float>&,
                                     const FwdInput&, const Op64&, const Reduce&, float*, int, int);
template void launch_yfft_inv<double>(hipStream_t, const Dims&, const FftPlan&, const Tables<double>&,
                                      const double*, double*, const Reduce&, int, int, bool);
template void launch_yfft_inv<float>(hipStream_t, const Dims&, const FftPlan&, const Tables<float>&,
                                     const float*, double*, const Reduce&, int, int, bool);

}  // namespace eddy
