// resident.hip -- kernels of the resident time loop: a substep's predicted velocity made
// on the device from the previous corrected one plus seeded noise, and the per-step log of
// the post-projection divergence range (what SCRINFO prints, info.f:5-165).
//
// Noise: three N(0,1) draws per cell from Philox4x32-10 (Salmon, Moraes, Dror, Shaw,
// "Parallel random numbers: as easy as 1, 2, 3", SC'11) with counter {cell lo, cell hi,
// step, 0} and key {seed, 0}, Box-Muller on words (0,1) and (2,3). `cell` is the 0-based
// offset of the cell in the DP(NX,NY,NZ) array and `step` is read from device memory, so a
// captured graph draws fresh noise on every replay.
#include "kernels.h"
#include "stencil_device.h"

namespace eddy {

struct Words {
    uint32_t w0, w1, w2, w3;
};

__device__ __forceinline__ Words philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3, uint32_t k0,
                                               uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        // one 32 x 32 -> 64-bit product per multiplier (a single v_mad_u64_u32) gives both halves
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        const uint32_t n0 = hi1 ^ c1 ^ k0;
        const uint32_t n2 = hi0 ^ c3 ^ k1;
        c1 = lo1;
        c3 = lo0;
        c0 = n0;
        c2 = n2;
        k0 += 0x9E3779B9u;
        k1 += 0xBB67AE85u;
    }
    return Words{c0, c1, c2, c3};
}

// The three functions of the Box-Muller step, on the arguments that it meets, each within about an
// ulp. The library's take any argument; these leave out what 33-bit fractions cannot need (ranges,
// denormals, general reductions) and share one polynomial between sine and cosine. The
// polynomials are minimax fits (Remez exchange) of the functions named beside them.

// sqrt(-2 ln u), u = (a + 1/2) 2^-32. With u = 2^k (1 + f), 1 + f in [sqrt 1/2, sqrt 2), and
// s = f / (2 + f): ln(1 + f) = 2 atanh(s) = f - (f^2/2 - s (f^2/2 + R(s^2))), where s R(s^2) is
// 2 atanh(s) - 2 s; f is exact, so the logarithm is accurate to its last bits near 1 too. What its
// rounding leaves over goes into the root's last correction.
__device__ __forceinline__ double radius(uint32_t a) {
    const double x = (double)a + 0.5;
    const int hx = __double2hiint(x), mh = hx & 0xfffff;
    const bool up = mh >= 0x6a09e;  // mantissa above sqrt 2
    const double k = (double)((hx >> 20) - 1023 - 32 + (up ? 1 : 0));
    const double m = __hiloint2double(mh | (up ? 0x3fe00000 : 0x3ff00000), __double2loint(x));
    const double f = m - 1.0, d = m + 1.0;
    double r = __builtin_amdgcn_rcp(d);
    r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
    double s = f * r;
    s = __builtin_fma(__builtin_fma(-d, s, f), r, s);
    const double z = s * s;
    // (2 atanh(s)/s - 2)/s^2 on s^2 <= 0.0295, error below 2^-66 of the logarithm
    double p = 0.13251317387323894;
    p = __builtin_fma(p, z, 0.13250119327470272);
    p = __builtin_fma(p, z, 0.15387090709603735);
    p = __builtin_fma(p, z, 0.1818177566646405);
    p = __builtin_fma(p, z, 0.22222222646787104);
    p = __builtin_fma(p, z, 0.28571428569085927);
    p = __builtin_fma(p, z, 0.4000000000000625);
    p = __builtin_fma(p, z, 0.6666666666666666);
    const double h = 0.5 * f * f;
    // ln 2 in two parts, the first with 20 low zero bits: k times it is exact
    const double t = __builtin_fma(s, __builtin_fma(p, z, h), k * 7.440617110012397e-11);
    // x + xl = -ln u: the two leading terms summed exactly, then the small one
    const double c = k * -0.6931471804855391, s0 = c - f, sl = (c - s0) - f;
    const double w = sl + (h - t), x0 = s0 + w, xl = w - (x0 - s0);
    // the root of 2 (x0 + xl): Newton on the reciprocal root of 2 x0 (1e-10 < x0 < 23)
    const double x2 = 2.0 * x0, y = __builtin_amdgcn_rsq(x2);
    double g = x2 * y, q = 0.5 * y;
    const double e = __builtin_fma(-q, g, 0.5);
    g = __builtin_fma(g, e, g);
    q = __builtin_fma(q, e, q);
    return __builtin_fma(__builtin_fma(2.0, xl, __builtin_fma(-g, g, x2)), q, g);
}

// sin(pi w), |w| <= 1/2: 2.5 w + w (pi - 2.5 + w^2 P(w^2)). The slope 2.5 lies between the function's
// 2 and pi, so that the rounded second term stays below a quarter of the result.
__device__ __forceinline__ double sin_pi(double w) {
    const double z = w * w;
    double p = -2.2280551655931242e-08;
    p = __builtin_fma(p, z, 7.948506120737306e-07);
    p = __builtin_fma(p, z, -2.191524891736974e-05);
    p = __builtin_fma(p, z, 0.0004663027871623419);
    p = __builtin_fma(p, z, -0.007370430943669141);
    p = __builtin_fma(p, z, 0.08214588661099206);
    p = __builtin_fma(p, z, -0.5992645293207869);
    p = __builtin_fma(p, z, 2.5501640398773455);
    p = __builtin_fma(p, z, -5.16771278004997);
    return __builtin_fma(w, 2.5, w * __builtin_fma(p, z, 0.6415926535897932));
}

// The angle 2 pi (b + 1/2) 2^-32 as pi (y + 1), y in (-1, 1) exact: its cosine is -sin(pi h) with
// h = 1/2 - |y|, its sine -sign(y) sin(pi (1/2 - |h|)).
__device__ __forceinline__ double angle_y(uint32_t b) {
    return __builtin_fma((double)b, 0x1p-31, 0x1p-32 - 1.0);
}

// Both deviates of a pair.
__device__ __forceinline__ void box_muller(uint32_t a, uint32_t b, double& g0, double& g1) {
    const double r = radius(a), y = angle_y(b), h = 0.5 - fabs(y);
    g0 = -r * sin_pi(h);
    g1 = -r * copysign(sin_pi(0.5 - fabs(h)), y);
}

// The first deviate of a pair only.
__device__ __forceinline__ double box_muller_first(uint32_t a, uint32_t b) {
    return -radius(a) * sin_pi(0.5 - fabs(angle_y(b)));
}

// One thread per element of a plane, consecutive elements to consecutive lanes. Faces CORRECT updates
// get sigma * N(0,1) (U: I = 1..NX-3, V: all, W: K = 1..NZ-3, 0-based, over interior cells);
// periodic ghost rows J = 0, NY-1 take their images' values; the rest is copied. Bound by
// instruction issue beside its 48 B/cell: per cell ten Philox rounds of two quarter-rate 32 x 32-bit
// products, two logarithms and roots and three sine polynomials: 481 -> 259 vector instructions with the
// functions above in place of the library's log, sqrt, sincospi and cospi, and 1.010 -> 0.684 ms at
// 768 x 384 x 256 (5.3 TB/s). Their deviates are nearer to the exact ones: 0.535 ulp in the root mean
// square against 0.540, 2.39 at most against 2.45 (two million draws).
__global__ void __launch_bounds__(256) k_perturb(Dims d, const double* __restrict__ u, const double* __restrict__ v,
                                                 const double* __restrict__ w, double* __restrict__ us,
                                                 double* __restrict__ vs, double* __restrict__ ws, double sigma,
                                                 uint32_t seed, const int* __restrict__ step, unsigned rnx) {
    const unsigned pl = (unsigned)d.nx * (unsigned)d.ny, r = blockIdx.x * 256u + threadIdx.x;
    if (r >= pl) return;
    const int K = blockIdx.y;
    int J = (int)__umulhi(r, rnx);  // exact or one too large
    int I = (int)r - J * d.nx;
    if (I < 0) {
        --J;
        I += d.nx;
    }
    const size_t t = (size_t)pl * K + r;
    const bool inner = I >= 1 && I <= d.M && K >= 1 && K <= d.N;
    if (!inner) {
        us[t] = u[t];
        vs[t] = v[t];
        ws[t] = w[t];
        return;
    }
    const int Js = (J == 0) ? d.L : ((J == d.L + 1) ? 1 : J);
    const size_t o = sidx(d, I, Js, K);
    const double uo = u[I <= d.nx - 3 ? o : t], vo = v[o], wo = w[K <= d.nz - 3 ? o : t];
    const Words x = philox4x32_10((uint32_t)o, (uint32_t)(o >> 32), (uint32_t)step[0], 0u, seed, 0u);
    double g0, g1;
    box_muller(x.w0, x.w1, g0, g1);
    const double g2 = box_muller_first(x.w2, x.w3);  // the pair's second deviate is not used
    us[t] = (I <= d.nx - 3) ? uo + sigma * g0 : uo;
    vs[t] = vo + sigma * g1;
    ws[t] = (K <= d.nz - 3) ? wo + sigma * g2 : wo;
}

void launch_perturb(hipStream_t st, const Dims& d, const double* u, const double* v, const double* w, double* us,
                    double* vs, double* ws, double sigma, uint32_t seed, const int* step) {
    const dim3 grid((unsigned)(((size_t)d.nx * d.ny + 255) / 256), d.nz);
    hipLaunchKernelGGL(k_perturb, grid, dim3(256), 0, st, d, u, v, w, us, vs, ws, sigma, seed, step,
                       (unsigned)(((1ull << 32) + d.nx - 1) / d.nx));
}

}  // namespace eddy
