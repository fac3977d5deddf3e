// mma_device.h -- the 16 x 16 x 4 matrix-core products of the FP64 and FP32 kernels.
//
// Lane layout of run(a, b, c), D = A B + C with A 16 x 4, B 4 x 16: lane l supplies A(l%16, l/16)
// and B(l/16, l%16); accumulator element v of lane l is D(row(l/16, v), l%16). The f64 rows
// interleave across the four lane groups (checked on the device), the f32 rows do not.
#pragma once

#include "common.h"

namespace eddy {

template <typename T>
struct Mma;
template <>
struct Mma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 run(double a, double b, v4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return q + 4 * v; }
};
template <>
struct Mma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ v4 run(float a, float b, v4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int v) { return 4 * q + v; }
};

}  // namespace eddy
