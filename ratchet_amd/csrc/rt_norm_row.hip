// The 16-bit LayerNorm / RMSNorm with a wave per row (arithmetic contract: rt_norm.hip).
#include "rt_norm.h"
#include "rt_ordered.h"

namespace {

// ------------------------------------------------------------------------------------------------------------------
// LayerNorm / RMSNorm in the 16-bit types, one wave per row, the row in registers: the reference's sums without a walk.
//
// The reference adds x and T(x*x) left to right in f32 and rounds each sum to T once (cpu/norm.rs:72-89, half's Sum).  What is needed is
// therefore not the f32 sum but what it rounds to, and that is the same for almost every sum near it: this kernel adds in any order,
// bounds how far the ordered sum can be from that, and is done if both ends of the interval round to one value of T.
//   T(x*x): all terms are >= 0, so every rounding of the ordered sum, and of this one, is at most 2^-24 of the partial sum it rounds.  N(0, 1) rows
//        of 2560 columns stay open one in 35 in bf16, one in four in f16; a count of the terms that can make an add inexact at all halves
//        that in f16 and takes bf16 to a few in a thousand.
//   x: the sum of terms of both signs is small against its terms, but nearly all of its adds are exact: a term that is a multiple
//        of U, the ulp of the largest partial sum of the row, never makes an add inexact, and what one other term can make the sum lose, in its own add and
//        in those where the sum later grows into coarser binades, is at most u/2 + 2u/2 + 4u/2 + ... <= U.  The partial sums are bounded by a prefix
//        sum over the lanes and the largest partial sum inside a lane's vector.  That bound does not shrink with the sum, and what the sum rounds to
//        does: N(0, 1) rows of 2560 columns stay open one in a thousand, the same with their mean taken off one in six, rows whose sum is
//        zero but for the roundings on the way all of them (f16, of whose terms more are not multiples of U: one in fifty, all, all).
// Rows that stay open get the ordered sum itself (norm_ordered_squares, norm_ordered_sum), 2.5 and 3 us a wave for 2560 columns.
// What bounds it: memory where there are many rows ([16384,3072] bf16 RMSNorm 40.3 -> 36.9 us, a copy of its bytes 31.5), and in LayerNorm the vector
// instructions, of which it takes twenty an element (47 -> 41 us); where there are few, launch, loads and the rows that stay open
// ([256,2560] bf16 RMSNorm 14.3 -> 6.1 us).  A block is one wave: a row that takes longer then keeps no place but its own.
// ------------------------------------------------------------------------------------------------------------------
constexpr int NR_STREAM = 2;                                 // the non-temporal hint of a buffer access
constexpr int NR_BLOCK = 64;

// The f32 chain of 16-bit terms.  pair(a, b) starts two sums at two bit patterns, run() adds a vector's eight terms to both, lo() and hi() are the sums' bit patterns; one() adds to a single sum.
template <typename T> struct ChainF32;
template <> struct ChainF32<half_t> {
    struct Pair {
        float a, b;
    };
    static __device__ __forceinline__ Pair pair(uint32_t a, uint32_t b) { return Pair{u2f(a), u2f(b)}; }
    static __device__ __forceinline__ uint32_t lo(const Pair& p) { return f2u(p.a); }
    static __device__ __forceinline__ uint32_t hi(const Pair& p) { return f2u(p.b); }
    // 1.0 * widen(h) + sum, one instruction with one rounding
#define RT_MIX2(N)                                                              \
    "v_fma_mix_f32 %0, %" #N ", %6, %0 op_sel_hi:[1,0,0]\n"                      \
    "v_fma_mix_f32 %1, %" #N ", %6, %1 op_sel_hi:[1,0,0]\n"                      \
    "v_fma_mix_f32 %0, %" #N ", %6, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n"       \
    "v_fma_mix_f32 %1, %" #N ", %6, %1 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n"
    static __device__ __forceinline__ void run(Pair& p, const v4u& v) {
        const float one = 1.0f;
        asm(RT_MIX2(2) RT_MIX2(3) RT_MIX2(4) RT_MIX2(5) : "+v"(p.a), "+v"(p.b) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(one));
    }
#undef RT_MIX2
#define RT_MIX1(N)                                                              \
    "v_fma_mix_f32 %0, %" #N ", %5, %0 op_sel_hi:[1,0,0]\n"                      \
    "v_fma_mix_f32 %0, %" #N ", %5, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]\n"
    static __device__ __forceinline__ uint32_t one(uint32_t s, const v4u& v) {
        float a = u2f(s);
        const float one = 1.0f;
        asm(RT_MIX1(1) RT_MIX1(2) RT_MIX1(3) RT_MIX1(4) : "+v"(a) : "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "s"(one));
        return f2u(a);
    }
#undef RT_MIX1
};
template <> struct ChainF32<bf16_t> {
    struct Pair {
        float a, b;
    };
    static __device__ __forceinline__ Pair pair(uint32_t a, uint32_t b) { return Pair{u2f(a), u2f(b)}; }
    static __device__ __forceinline__ uint32_t lo(const Pair& p) { return f2u(p.a); }
    static __device__ __forceinline__ uint32_t hi(const Pair& p) { return f2u(p.b); }
    static __device__ __forceinline__ void run(Pair& p, const v4u& v) {
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float l = u2f(v[w] << 16), h = u2f(v[w] & 0xffff0000u);
            p.a += l;
            p.b += l;
            p.a += h;
            p.b += h;
        }
    }
    static __device__ __forceinline__ uint32_t one(uint32_t s, const v4u& v) {
        float a = u2f(s);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            a += u2f(v[w] << 16);
            a += u2f(v[w] & 0xffff0000u);
        }
        return f2u(a);
    }
};

template <typename T> struct NormVec;
template <> struct NormVec<half_t> {
    static constexpr float SPAN = 0x1p10f;                                       // a normal value over its ulp, at least
    static __device__ __forceinline__ void widen(const v4u& x, float (&f)[8]) {
        const np_h8 h = __builtin_bit_cast(np_h8, x);
#pragma unroll
        for (int q = 0; q < 8; q++) f[q] = (float)h[q];
    }
    static __device__ __forceinline__ v4u square(const v4u& x) {                 // T(x*x): eight f16 products, each rounded once
        const np_h8 h = __builtin_bit_cast(np_h8, x);
        return __builtin_bit_cast(v4u, h * h);
    }
    static __device__ __forceinline__ float squares(const v4u& x, const float (&)[8]) { return u2f(ChainF32<half_t>::one(0, square(x))); }
    // how many of the wave's elements are below `bound` in magnitude (or a little above it)
    static __device__ __forceinline__ uint32_t below(const v4u& x, float bound) {
        const np_h8 h = __builtin_bit_cast(np_h8, x);
        const half_t b = (half_t)(bound * (1.0f + 0x1p-9f) + 0x1p-24f);
        uint32_t n = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(__builtin_fabsf16(h[q]) < b));
        return n;
    }
};
template <> struct NormVec<bf16_t> {
    static constexpr float SPAN = 0x1p7f;
    static __device__ __forceinline__ void widen(const v4u& x, float (&f)[8]) {
#pragma unroll
        for (int w = 0; w < 4; w++) {
            f[2 * w] = u2f(x[w] << 16);
            f[2 * w + 1] = u2f(x[w] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ v4u square(const v4u& x) {
        float f[8];
        widen(x, f);
        v4u out;
#pragma unroll
        for (int w = 0; w < 4; w++) asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(out[w]) : "v"(f[2 * w] * f[2 * w]), "v"(f[2 * w + 1] * f[2 * w + 1]));
        return out;
    }
    static __device__ __forceinline__ float squares(const v4u&, const float (&f)[8]) {
        float acc = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; q++) acc += np_round_bf16(f[q] * f[q]);
        return acc;
    }
    static __device__ __forceinline__ uint32_t below(const v4u& x, float bound) {
        const float more = bound * (1.0f + 0x1p-6f);         // (for the low half under a word's high one)
        uint32_t n = 0;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(fabsf(u2f(x[w] << 16)) < more));
            n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(fabsf(u2f(x[w])) < more));
        }
        return n;
    }
};

// the sum of eight terms, left to right, and the largest magnitude of a partial sum
__device__ __forceinline__ float nr_partial(const float (&f)[8], float& top) {
    float s = f[0], m = fabsf(s);
#pragma unroll
    for (int q = 1; q < 8; q++) {
        s += f[q];
        m = fmaxf(m, fabsf(s));
    }
    top = m;
    return s;
}
// x, scale, bias and y on 16-byte boundaries, cols a multiple of 8 and at most 512 * V; a block to a row.
template <typename T, int V, int KIND>
__global__ void __launch_bounds__(NR_BLOCK) norm16_row_kernel(const T* x, const T* __restrict__ scale, const T* __restrict__ bias, T* y,
                                                              uint32_t cols, float eps) {
    __shared__ v4u park[V * 64];
    const uint32_t lane = threadIdx.x;
    const uint64_t row = blockIdx.x;
    const uint32_t nvec = cols / 8;
    const uint32_t pads = (V * 64 - nvec) * 8;               // zeros past the row's end: +0 terms change no sum
    // buffer accesses: where the row has ended a load gives zeros and a store is dropped, without a branch for each
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x) + row * cols, 0, cols * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y + row * cols, 0, cols * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(scale), 0, cols * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(bias ? bias : scale), 0, bias ? cols * 2 : 0, 0x00020000);
    v4u v[V];
#pragma unroll
    for (int j = 0; j < V; j++) v[j] = __builtin_amdgcn_raw_buffer_load_b128(rx, (j * 64 + lane) * 16, 0, NR_STREAM);
    // the squares' partial sums in step j are at most the total of the steps up to it: `area` bounds the sum of all of them
    float sq = 0.0f, area = 0.0f;
    float carry = 0.0f, reach = 0.0f, run = 0.0f;        // of x: the sum of the steps before; the largest partial sums of the row and of a vector
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < V; j++) {
        float f[8], top;
        NormVec<T>::widen(v[j], f);
        const float t = NormVec<T>::squares(v[j], f);
        sq += t;
        area += (float)(V - j) * t;
        if constexpr (KIND == NORM_LAYER) {
            const float part = nr_partial(f, top);
            const float upto = lanes_scan(part);
            reach = fmaxf(reach, fabsf(carry + lane_before(upto)) + top);
            run = fmaxf(run, top);
            carry += u2f(lane_value(f2u(upto), 63));
            sum += (double)part;
        }
        if (V > 8) __builtin_amdgcn_sched_barrier(0);        // (rows of 9 and 10 steps: one after the other, for fewer registers)
    }
    // (the widened values of one pass over the row are not to be held for the next: they are twice the registers of the row)
    auto forget = [&]() {
#pragma unroll
        for (int j = 0; j < V; j++) asm volatile("" : "+v"(v[j]));
    };
    forget();
    auto sure = [](float low, float high) -> bool {
        return __builtin_bit_cast(uint16_t, Ar<T>::conv(low)) == __builtin_bit_cast(uint16_t, Ar<T>::conv(high));
    };
    sq = wave_sum(sq);
    area = wave_sum(area);
    const float slack = (512.0f * area + (float)(V + 32) * sq) * 0x1.01p-24f;
    // (the same in all lanes, which the compiler does not know)
    uint32_t open = __builtin_amdgcn_readfirstlane(!sure(sq - slack, sq + slack));
    if (open) {
        // closer: a square has no bit SPAN times below its own size, so that those of SPAN times the sum's last ulp and up make no
        // add inexact.  Half an ulp for each of the others, one for what is left over where the sum passes into another
        // binade, and this sum's own roundings.
        const float u = nr_ulp(sq * (1.0f + 0x1p-7f)), small = __builtin_sqrtf(u * NormVec<T>::SPAN);
        uint32_t count = 0;
#pragma unroll
        for (int j = 0; j < V; j++) count += NormVec<T>::below(v[j], small);
        count -= pads;
        const float close = ((float)count * 0.5f + 1.0f) * u + (float)(8 * V + 32) * 0x1.01p-24f * sq;
        open = __builtin_amdgcn_readfirstlane(!(sq > 0x1p-60f && sq < 0x1p100f && sure(sq - close, sq + close)));
        forget();
    }
    float sx = 0.0f;
    if constexpr (KIND == NORM_LAYER) {
        // (1 + 2^-7: what the prefix sums, and the ordered sum itself, can be off by)
        reach = wave_max(reach) * (1.0f + 0x1p-7f);
        run = wave_max(run);
        sum = wave_sum(sum);
        const float u = nr_ulp(reach);
        uint32_t odd = 0;                                // terms that may not be multiples of u
#pragma unroll
        for (int j = 0; j < V; j++) odd += NormVec<T>::below(v[j], u * NormVec<T>::SPAN);
        odd -= pads;
        // a vector's sum of seven adds is off by half an ulp of its partial sums each, and only in vectors with such terms
        const double off = (double)odd * ((double)u + 4.0 * (double)nr_ulp(run)) + (double)u;
        sx = (float)sum;
        if (!(reach >= 0x1p-90f && reach < 0x1p100f && sure((float)(sum - off), (float)(sum + off)))) open |= reach == 0.0f ? 0 : 2;
    }
    forget();
    open = __builtin_amdgcn_readfirstlane(open);
    if (__builtin_expect(open != 0, 0)) {
        // (through LDS, in the lane that reads it again: a loop over the steps, not one piece of code for each; the steps of a
        // group side by side, and what was gained by it, cost more in LDS and registers, which keep other rows waiting)
#pragma unroll
        for (int j = 0; j < V; j++) park[j * 64 + lane] = v[j];
        const uint32_t steps = (nvec + 63) / 64;
        uint32_t s2 = 0;
        float s1 = 0.0f;
        v4u next = park[lane];
#pragma unroll 1
        for (uint32_t j = 0; j < steps; j++) {
            const v4u here = next;
            next = park[(j + 1 < steps ? j + 1 : j) * 64 + lane];
            if (KIND == NORM_LAYER && (open & 2)) s1 = norm_ordered_sum<NormVec<T>>(s1, here, lane);
            if (open & 1) s2 = norm_ordered_squares<ChainF32<T>>(s2, NormVec<T>::square(here), lane);
        }
#pragma unroll
        for (int j = 0; j < V; j++) v[j] = park[j * 64 + lane];      // (not in registers meanwhile)
        if (open & 1) sq = u2f(s2);
        if (open & 2) sx = s1;
    }
    const RowStats<T> st = finish_stats<T, KIND>(sx, sq, cols, eps);
    const uint32_t none = bias ? 0u : 0x80008000u;           // without a bias -0, which adds nothing
#pragma unroll
    for (int j = 0; j < V; j++) {
        const uint32_t at = (j * 64 + lane) * 16;
        const v4u sc = __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0);
        v4u bi = {0, 0, 0, 0};
        if (KIND == NORM_LAYER) {
            bi = __builtin_amdgcn_raw_buffer_load_b128(rb, at, 0, 0);
#pragma unroll
            for (int w = 0; w < 4; w++) bi[w] |= none;
        }
        __builtin_amdgcn_raw_buffer_store_b128(norm_vec16<T, KIND>(v[j], st, sc, bi), ry, at, 0, NR_STREAM);
    }
}

template <typename T, int KIND>
int launch_norm16_row(rt_device* dev, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols, float eps) {
    RT_REQUIRE(rows <= NR_MAX_ROWS, RT_ERR_SIZE, "norm: too many rows");
#define RT_NR(VC)                                                                                                                    \
    case VC:                                                                                                                         \
        hipLaunchKernelGGL((norm16_row_kernel<T, VC, KIND>), dim3((unsigned)rows), dim3(NR_BLOCK), 0, dev->stream, (const T*)x,      \
                           (const T*)scale, (const T*)bias, (T*)y, cols, eps);                                                       \
        break
    switch ((cols + 511) / 512) {
        RT_NR(1); RT_NR(2); RT_NR(3); RT_NR(4); RT_NR(5); RT_NR(6); RT_NR(7); RT_NR(8); RT_NR(9); RT_NR(10);
        default: return rt_fail(RT_ERR_ARG, "norm: internal: %u columns in the wave-per-row norm", cols);
    }
#undef RT_NR
    RT_CHECK_LAUNCH("norm16_row_kernel");
    return RT_OK;
}

}  // namespace

int rt_norm16_row(rt_device* dev, bool bf16, int kind, const void* x, const void* scale, const void* bias, void* y, uint64_t rows, uint32_t cols,
                  float eps) {
    if (kind == NORM_LAYER)
        return bf16 ? launch_norm16_row<bf16_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps)
                    : launch_norm16_row<half_t, NORM_LAYER>(dev, x, scale, bias, y, rows, cols, eps);
    return bf16 ? launch_norm16_row<bf16_t, NORM_RMS>(dev, x, scale, nullptr, y, rows, cols, eps)
                : launch_norm16_row<half_t, NORM_RMS>(dev, x, scale, nullptr, y, rows, cols, eps);
}
