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

#include "batch_device.h"
#include "kernels.h"
#include "xsolve_device.h"

namespace eddy {

// One block of 256/P lines (logical line block `lb`), 64/P lines per wave.
template <typename T, int QMAX, int ROWS, bool CYC = false>
__device__ __forceinline__ void xsolve_tile(const XArgs<T>& a, int lb) {
    extern __shared__ unsigned char smem_raw[];
    constexpr bool FIXED = ROWS != XR_ANY, PADDED = ROWS == XR_PADDED;
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
    // together. Every slot that a lane reads as a row of its line is written, also for lanes without a
    // line: their results are not stored, but the reduction's wrapped shuffles carry their values, times
    // 0, into the lines that are there, so those must be finite. Elements past the last line take the
    // last one's value; in the padded layout, where they fall elsewhere, a lane without a line zeroes
    // its own rows.
    T* const blk = a.S + (size_t)line0 * (size_t)M;
    const int nel = nl * M;
    const int wi = lane + (lane >> 3);
    // PADDED (LW <= 4): where element el of the wave's lines lies when each takes P*Q elements, so that a
    // lane's rows are Q consecutive ones as in an exact split (slots past M hold no row of the line)
    const int pad = P * Q - M;
    auto place = [&](int el) {
        int e = el;
        if (LW > 1) e += el >= M ? pad : 0;
        if (LW > 2) e += (el >= 2 * M ? pad : 0) + (el >= 3 * M ? pad : 0);
        return e + (e >> 3);
    };
    {
        T v[QMAX];
        if (PADDED && nl == LW) {  // M > P (Q - 1): only the last round reaches past the lines
#pragma unroll
            for (int u = 0; u < QMAX - 1; ++u) v[u] = blk[lane + 64 * u];
            v[QMAX - 1] = blk[min(lane + 64 * (QMAX - 1), nel - 1)];
        } else if (nel == 64 * QMAX) {  // wave-uniform
#pragma unroll
            for (int u = 0; u < QMAX; ++u) v[u] = blk[lane + 64 * u];
        } else {
#pragma unroll
            for (int u = 0; u < QMAX; ++u)
                v[u] = ld_off(blk, (unsigned)sizeof(T) * (unsigned)min(lane + 64 * u, nel - 1));
        }
#pragma unroll
        for (int u = 0; u < QMAX; ++u)
            if (PADDED) {
                if (lane + 64 * u < nel) tile[place(lane + 64 * u)] = v[u];
            } else if (FIXED || u < Q) {
                tile[wi + 72 * u] = v[u];
            }
        if (PADDED && nl < LW && lane >= nl * P) {
            const int e0 = lane * QMAX;
#pragma unroll
            for (int r = 0; r < QMAX; ++r) tile[e0 + r + ((e0 + r) >> 3)] = T(0);
        }
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
    T part = xsolve_lines<T, QMAX, ROWS, CYC>(
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
    if (PADDED) {
#pragma unroll
        for (int u = 0; u < QMAX; ++u)
            if (lane + 64 * u < nel)
                st_off(blk, (unsigned)sizeof(T) * (unsigned)(lane + 64 * u), tile[place(lane + 64 * u)]);
    } else if (nel == 64 * QMAX) {
#pragma unroll
        for (int u = 0; u < QMAX; ++u) blk[lane + 64 * u] = tile[wi + 72 * u];
    } else {
#pragma unroll
        for (int u = 0; u < QMAX; ++u)
            if (lane + 64 * u < nel) st_off(blk, (unsigned)sizeof(T) * (unsigned)(lane + 64 * u), tile[wi + 72 * u]);
    }
}

// Each XCD walks its lines from the last to the first, against the order of the x2 transforms on both
// sides: every pass then starts on what the pass before it left in the caches. The eighth of the lines
// that an XCD takes is the eighth of the x2 transforms' tiles that it took, so that spectra that fit the
// L2s are found there (128 x 128 x 128, 17 MB: this solve 0.0137 ms and the inverse x2 transform 0.0139; 0.0167 and
// 0.0137 in forward order; 0.0205 and 0.0204 where reversing the whole order gives an XCD another's eighth), and
// larger ones in the memory-side cache (768 x 384 x 256, 604 MB: 0.284 instead of 0.310 in forward order and
// 0.369 instead of 0.387).
template <typename T, int QMAX, int ROWS, bool CYC>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && ROWS != XR_ANY ? (QMAX <= 8 ? 6 : 4) : 1)))
k_xsolve(XArgs<T> a) {
    xsolve_tile<T, QMAX, ROWS, CYC>(a, xcd_tile_back(blockIdx.x, gridDim.x));
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
    xsolve_dispatch(xsolve_class(d.M, P, Q, cyc != 0), [&](auto qmax, auto rows) {
        constexpr int ROWS = decltype(rows)::value;
        auto go = [&](auto fn) {
            (void)hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sh);
            hipLaunchKernelGGL(fn, grid, dim3(256), sh, st, a);
        };
        if constexpr (ROWS != XR_ANY) go(k_xsolve<T, decltype(qmax)::value, ROWS, false>);
        else if (cyc) go(k_xsolve<T, decltype(qmax)::value, XR_ANY, true>);
        else go(k_xsolve<T, decltype(qmax)::value, XR_ANY, false>);
    });
    return 0;
}

// ------------------------------------------------------------------ batched (one item per workgroup)
// One kernel per rows-per-thread template: a kernel holding every template would take the
// registers of the largest (QMAX = 32) for all problems.
// Bounds where the unbounded kernel sits just above an occupancy step (8 rows: 86 VGPRs, 6 waves
// per SIMD at 80; 16 rows: 148, 4 waves at 128).
template <typename T, int QMAX, int ROWS>
__global__ void __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && ROWS != XR_ANY ? (QMAX <= 8 ? 6 : 4) : 1)))
k_batch_xsolve(const Job<XArgs<T>>* jobs, int njobs, int total) {
    run_item(jobs, njobs, total, [](const Job<XArgs<T>>& J, int t) { xsolve_tile<T, QMAX, ROWS>(J.a, t); });
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
        if (x.cls % kExact != y.cls % kExact) return x.cls % kExact > y.cls % kExact;
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
        xsolve_dispatch(sl.cls_q[c], [&](auto qmax, auto rows) {
            auto fn = k_batch_xsolve<T, decltype(qmax)::value, decltype(rows)::value>;
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
