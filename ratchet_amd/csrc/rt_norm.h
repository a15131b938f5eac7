// What the LayerNorm / RMSNorm kernels share: a row's statistics in the element type's arithmetic and what they make of an element.
#ifndef RT_NORM_H
#define RT_NORM_H

#include <type_traits>

#include "rt_arith.h"
#include "rt_internal.h"

namespace {

typedef _Float16 np_h8 __attribute__((ext_vector_type(8)));

enum { NORM_LAYER = 0, NORM_RMS = 1 };

// per-row statistics in T arithmetic, given f32 sums
template <typename T> struct RowStats {
    T mu, r;
};
template <typename T, int KIND> __device__ __forceinline__ RowStats<T> finish_stats(float sum_x, float sum_sq, uint32_t cols, float eps) {
    typedef Ar<T> A;
    RowStats<T> st;
    const T n = A::conv((float)cols);                       // T::from(step as f32)
    const T x2 = A::div(A::conv(sum_sq), n);
    T var;
    if (KIND == NORM_LAYER) {
        st.mu = A::div(A::conv(sum_x), n);
        var = A::sub(x2, A::mul(st.mu, st.mu));
    } else {
        st.mu = A::conv(0.0f);
        var = x2;
    }
    const T t = A::add(var, A::conv(eps));
    st.r = A::div(A::conv(1.0f), ar_sqrt<T>(t));
    return st;
}

template <typename T, int KIND> __device__ __forceinline__ T norm_one(T x, const RowStats<T>& st, T scale, T bias, bool has_bias) {
    typedef Ar<T> A;
    T v = (KIND == NORM_LAYER) ? A::sub(x, st.mu) : x;
    v = A::mul(v, st.r);
    v = A::mul(v, scale);
    if (KIND == NORM_LAYER && has_bias) v = A::add(v, bias);
    return v;
}

// f rounded to bf16 and widened again, in one instruction: converted into the high half of a word whose low half is bf16(0) = 0
__device__ __forceinline__ float np_round_bf16(float f) {
    uint32_t r;
    asm("v_cvt_pk_bf16_f32 %0, 0, %1" : "=v"(r) : "v"(f));
    return u2f(r);
}
// norm_one, with a bias, on the eight elements of a vector.  bf16 goes in f32 form from step to step, two instructions each (through
// Ar<bf16_t> the roundings and widenings take four), and is packed once at the end.
template <typename T, int KIND> __device__ __forceinline__ v4u norm_vec16(const v4u& x, const RowStats<T>& st, const v4u& scale, const v4u& bias) {
    v4u out;
    if constexpr (std::is_same<T, bf16_t>::value) {
        const float mu = Ar<T>::widen(st.mu), rs = Ar<T>::widen(st.r);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            float v[2] = {u2f(x[w] << 16), u2f(x[w] & 0xffff0000u)};
            const float s[2] = {u2f(scale[w] << 16), u2f(scale[w] & 0xffff0000u)}, b[2] = {u2f(bias[w] << 16), u2f(bias[w] & 0xffff0000u)};
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (KIND == NORM_LAYER) v[h] = np_round_bf16(v[h] - mu);
                v[h] = np_round_bf16(v[h] * rs) * s[h];
                if (KIND == NORM_LAYER) v[h] = np_round_bf16(v[h]) + b[h];
            }
            asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(out[w]) : "v"(v[0]), "v"(v[1]));
        }
    } else {
        np_h8 v = __builtin_bit_cast(np_h8, x);
        if (KIND == NORM_LAYER) v = v - st.mu;
        v = v * st.r * __builtin_bit_cast(np_h8, scale);
        if (KIND == NORM_LAYER) v = v + __builtin_bit_cast(np_h8, bias);
        out = __builtin_bit_cast(v4u, v);
    }
    return out;
}
}  // namespace

#endif
