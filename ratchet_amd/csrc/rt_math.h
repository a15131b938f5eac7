// Device math used by the elementwise / softmax / norm kernels: the libm-level routines (rt_libm.h, shared with the host
// check), 16-bit helpers and the wave / row reductions.  Compile with -ffp-contract=off.
#ifndef RT_MATH_H
#define RT_MATH_H

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// n / d in rt_tanhf: the reciprocal, the quotient, one correction by the exact remainder.  Four instructions where the
// general division takes ten, which also refine the reciprocal, scale the operands and put the special cases right.
// This is not correctly rounded for every pair of operands, but rt_tanhf's two divisions see only the pairs that its 2^32
// arguments lead to: d is in [1, 2^64], so the reciprocal is a normal float, and a quotient in the subnormal range or zero
// comes with d = 2 and an n that is twice a float (-em1 for |x| below 2^-25), so it is exact.
// With v_rcp_f32 anywhere within its one ulp all results equal the C library's but for 113 arguments of either sign, whose
// second quotient hangs on the reciprocal's last bit: tests/device_math_check.cpp finds them on the CPU, and
// test_tanh_where_the_division_hangs_on_the_reciprocal holds this chip's results on them to the C library's.
__device__ __forceinline__ float rt_div_mid(float n, float d) {
    const float r = __builtin_amdgcn_rcpf(d);
    const float q = n * r;
    return __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q);
}

#define RT_FN __device__ inline
#define RT_TABLE __device__ static const
#define RT_DIV(n, d) rt_div_mid(n, d)
#define RT_MED3(v, lo, hi) __builtin_amdgcn_fmed3f(v, lo, hi)
#include "rt_libm.h"
#undef RT_FN
#undef RT_TABLE
#undef RT_DIV
#undef RT_MED3

// ---- 16-bit helpers -------------------------------------------------------------------------------------
__device__ __forceinline__ float h2f(half_t h) { return (float)h; }
__device__ __forceinline__ half_t f2h(float f) { return (half_t)f; }              // round to nearest even
__device__ __forceinline__ uint16_t h_bits(half_t h) { return __builtin_bit_cast(uint16_t, h); }
__device__ __forceinline__ half_t bits_h(uint16_t u) { return __builtin_bit_cast(half_t, u); }

// ---- wave64 reductions ----------------------------------------------------------------------------------
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    return v;
}

// Reduction over the LANES threads that share a row: a group of 2..64 neighbouring lanes of a wave (a butterfly over the
// group; LANES == 64 is the whole wave), or a whole 256-thread block, whose four wave results meet in LDS and are added
// in a fixed order.  Every thread of the block must call the block form.
template <int LANES> __device__ __forceinline__ float row_sum(float v) {
    if constexpr (LANES <= 64) {
#pragma unroll
        for (int off = LANES / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    } else {
        v = wave_sum(v);
        __shared__ float red[LANES / 64];
        __syncthreads();                                   // earlier readers of red are done
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        v = red[0];
#pragma unroll
        for (int w = 1; w < LANES / 64; w++) v += red[w];
    }
    return v;
}
template <int LANES> __device__ __forceinline__ float row_max(float v) {
    if constexpr (LANES <= 64) {
#pragma unroll
        for (int off = LANES / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
    } else {
        v = wave_max(v);
        __shared__ float red[LANES / 64];
        __syncthreads();
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        v = red[0];
#pragma unroll
        for (int w = 1; w < LANES / 64; w++) v = fmaxf(v, red[w]);
    }
    return v;
}

#endif
