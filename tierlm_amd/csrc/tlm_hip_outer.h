/* tlm_hip_outer.h - rounded float products of a tile from the matrix cores:
 * v_mfma_f32 with K = 1 and C = 0 gives the outer product of ROWS values and 64
 * values with v_mul_f32's rounding, for chains that need a rounded product and
 * then a rounded add (an fma would round once).  Subnormals, infinities and NaNs
 * are v_mul_f32's; a product that is exactly -0 comes out as +0 (-0 + C), which
 * no chain here can show: each starts at +0, a sum of +0 and either zero is +0,
 * and no sum of others is -0.  The start-up self-test compares every shape with
 * v_mul_f32.  Included by .hip files. */
#ifndef TLM_HIP_OUTER_H
#define TLM_HIP_OUTER_H

#include "tlm_hip_internal.h"

/* lane l gives the value of row l % ROWS and of column l, and holds ROWS of the
 * products: element v is of row(v, l) and column col(v, l), elements v and
 * v + RV of one row */
template <int ROWS> struct Outer;
template <> struct Outer<32> {
    static constexpr int RV = 16;
    typedef float T __attribute__((ext_vector_type(32)));
    static __device__ __forceinline__ T mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, T{}, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int lane) { return 8 * ((v >> 2) & 3) + 4 * (lane >> 5) + (v & 3); }
    static __device__ __forceinline__ int col(int v, int lane) { return 32 * (v >> 4) + (lane & 31); }
};
template <> struct Outer<16> {
    static constexpr int RV = 4;
    typedef float T __attribute__((ext_vector_type(16)));
    static __device__ __forceinline__ T mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, T{}, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int lane) { return 4 * (lane >> 4) + (v & 3); }
    static __device__ __forceinline__ int col(int v, int lane) { return 16 * (v >> 2) + (lane & 15); }
};
template <> struct Outer<4> {
    static constexpr int RV = 4;
    typedef f32x4 T;
    static __device__ __forceinline__ T mul(float a, float b) {
        return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, T{}, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int v, int) { return v; }
    static __device__ __forceinline__ int col(int, int lane) { return lane; }
};

#endif
