// MFMA operand and result layouts of the 16 x 16 x 4 instructions on gfx950.
#pragma once

#include "tags_common.h"

namespace tags {

template <typename T>
struct Mfma;
// 16x16x4 blocks; lane l supplies A[l%16][l/16] and B[l/16][l%16]. Result
// element v of lane l is D[row(l, v)][l%16] with row = l/16 + 4v for the f64
// instruction and 4(l/16) + v for the f32 one (measured on gfx950).
template <>
struct Mfma<double> {
    typedef double v4 __attribute__((ext_vector_type(4)));
    static __device__ inline v4 run(double a, double b, v4 c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mfma<float> {
    typedef float v4 __attribute__((ext_vector_type(4)));
    static __device__ inline v4 run(float a, float b, v4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

}  // namespace tags
