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
// One butterfly step: the value of the lane whose index differs in bit OFF, joined with this lane's by `f` (commutative).  32 and 16 are
// register swaps of half waves and of rows of 16 lanes, the rest DPP moves inside a row, without the trip through LDS of a
// shuffle (about 60 cycles a step, six steps a reduction).  8 and 4 rotate a row of 16: the same partner, or after the steps before one that
// holds the same value, so 4 needs the step of 8 before it (groups of 8 lanes and fewer take the shuffle there).
template <int OFF, bool ROW, typename F> __device__ __forceinline__ float wave_step(float v, F f) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    if constexpr (OFF == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
        return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
    } else if constexpr (OFF == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
        return f(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
    } else if constexpr (OFF == 4 && !ROW) {
        return f(v, __shfl_xor(v, 4, 64));
    } else {
        constexpr int CTRL = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4E : 0xB1;      // row_ror:8, row_ror:4, quad_perm 2301, 1032
        const int o = __builtin_amdgcn_update_dpp(0, (int)u, CTRL, 0xf, 0xf, false);
        return f(v, __builtin_bit_cast(float, o));
    }
}
template <int LANES, typename F> __device__ __forceinline__ float lanes_join(float v, F f) {
    if constexpr (LANES >= 64) v = wave_step<32, true>(v, f);
    if constexpr (LANES >= 32) v = wave_step<16, true>(v, f);
    if constexpr (LANES >= 16) v = wave_step<8, true>(v, f);
    if constexpr (LANES >= 8) v = wave_step<4, (LANES >= 16)>(v, f);
    if constexpr (LANES >= 4) v = wave_step<2, true>(v, f);
    if constexpr (LANES >= 2) v = wave_step<1, true>(v, f);
    return v;
}
struct JoinSum { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
struct JoinMax { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
__device__ __forceinline__ float wave_sum(float v) { return lanes_join<64>(v, JoinSum()); }
// the same butterfly on doubles, whose two halves move side by side
template <int OFF> __device__ __forceinline__ double wave_step_sum(double v) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    uint32_t a[2], b[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const uint32_t w = (uint32_t)(u >> (32 * k));
        if constexpr (OFF >= 16) {
            const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(w, w, false, false) : __builtin_amdgcn_permlane16_swap(w, w, false, false);
            a[k] = r[0];
            b[k] = r[1];
        } else {
            constexpr int CTRL = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4E : 0xB1;
            a[k] = w;
            b[k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, CTRL, 0xf, 0xf, false);
        }
    }
    return __builtin_bit_cast(double, (uint64_t)a[1] << 32 | a[0]) + __builtin_bit_cast(double, (uint64_t)b[1] << 32 | b[0]);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = wave_step_sum<32>(v);
    v = wave_step_sum<16>(v);
    v = wave_step_sum<8>(v);
    v = wave_step_sum<4>(v);
    v = wave_step_sum<2>(v);
    return wave_step_sum<1>(v);
}
__device__ __forceinline__ float wave_max(float v) { return lanes_join<64>(v, JoinMax()); }

// Reduction over the LANES threads that share a row: a group of 2..64 neighbouring lanes of a wave (a butterfly over the
// group; LANES == 64 is the whole wave), or a whole 256-thread block, whose four wave results meet in LDS and are added
// in a fixed order.  Every thread of the block must call the block form.
template <int LANES> __device__ __forceinline__ float row_sum(float v) {
    if constexpr (LANES <= 64) {
        v = lanes_join<LANES>(v, JoinSum());
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
        v = lanes_join<LANES>(v, JoinMax());
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
