// mfma.hpp -- the 16x16x4 FP64 / FP32 matrix instructions and their layouts
// (wave64): A: lane l holds A[l%16][l/16]; B: lane l holds B[l/16][l%16]; D:
// lane l, register v holds D[row][l%16] with row = Mfma<T>::row(l, v) (FP64:
// l/16 + 4v, measured on gfx950; FP32: 4(l/16) + v).
#pragma once

#include "common.hpp"

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
template <>
struct Mfma<double>
{
    typedef dbl4 acc;
    static __device__ inline acc op(double a, double b, acc c)
    {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct Mfma<float>
{
    typedef flt4 acc;
    static __device__ inline acc op(float a, float b, acc c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ inline int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

// chunks of 16 points per FP32 accumulation chain
#define CT_FLUSH 4
