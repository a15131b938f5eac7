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
//        sum over the lanes and the largest partial sum inside a lane's vector.  N(0, 1) rows of 2560 columns stay open one in fifty in f16, one in
//        a thousand in bf16.
// Rows that stay open get the ordered sum itself (norm_ordered_squares, norm_ordered_sum), 2.5 and 4 us a wave for 2560 columns.
// What bounds it: memory where there are many rows ([16384,3072] bf16 RMSNorm 40.3 -> 36.9 us, a copy of its bytes 31.5), and in LayerNorm the vector
// instructions, of which bf16 takes twenty an element (47 -> 41 us); where there are few, launch, loads and the rows that stay open
// ([256,2560] bf16 RMSNorm 14.3 -> 6.1 us).  A block is one wave: a row that takes longer then keeps no place but its own.
// ------------------------------------------------------------------------------------------------------------------
constexpr int NR_STREAM = 2;                                 // the non-temporal hint of a buffer access
constexpr int NR_BLOCK = 64;

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

// the ulp of the binade of m (m finite, at least 2^-103; zero below that)
__device__ __forceinline__ float nr_ulp(float m) {
    const uint32_t e = f2u(m) >> 23;
    return e > 23 ? u2f((e - 23) << 23) : 0.0f;
}
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
// what f, a value of a 16-bit type, is off the nearest multiple of u = magic * 2^-23 / 1.5, a power of two or zero: zero, or NaN for inf and
// NaN, if it is none.  (Up to 2^22 u the sum has the ulp u; values beyond 2^11 u have no bit below u.)
__device__ __forceinline__ float nr_off(float f, float magic) {
    return f - ((f + magic) - magic);
}

// Both ordered sums take a step of 512 columns, 64 vectors, one a lane.
//
// x's: up to a lane the sum runs exactly, and is q (in double), as long as the lanes before it are `easy`: their terms and their q are
// multiples of the ulp of the binade that their partial sums stay in.  The first lane that is not easy adds its eight terms to the exact
// sum for real, and the lanes behind it start from there.
template <typename T>
__device__ __forceinline__ float norm_ordered_sum(float s, const v4u& x, uint32_t lane) {
    float f[8], part = 0.0f, low = 0.0f, high = 0.0f;        // a lane's sum, the ends of its partial sums
    NormVec<T>::widen(x, f);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        part += f[k];
        low = fminf(low, part);
        high = fmaxf(high, part);
    }
    const float guess = s + lane_before(lanes_scan(part)), near = fmaxf(guess + high, -(guess + low));       // (nothing rests on the guess)
    const float ulp = nr_ulp(near), coarse = nr_ulp(u2f(__builtin_amdgcn_readfirstlane(f2u(wave_max(near)))));
    float rest = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; k++) rest += fabsf(nr_off(f[k], ulp * 0x1.8p23f));
    // (terms far below the coarsest ulp would not be exact in the doubles either: such lanes add for real)
    const bool plain = (ulp > 0.0f) & (ulp >= coarse * 0x1p-20f) & (coarse < 0x1p100f) & (rest == 0.0f);
    const double mine = plain ? (double)part : 0.0, upto = lanes_scan(mine), before = upto - mine;
    const double limit = (double)ulp * 0x1p24, magic = (double)ulp * 0x1.8p52;       // sums up to the limit in steps of ulp are f32 values
    const double above = limit - (double)high, below = -limit - (double)low;
    const double grid = (double)coarse * 0x1.8p30;           // multiples of coarse * 2^-22
    double off = (double)s;                                  // the running sum less `before`, or, odd, what a double cannot hold:
    bool odd = !((off + grid) - grid == off);                // then the next lane adds to s itself
    for (uint32_t from = 0; from < 64;) {
        const double q = off + before;
        const bool easy = plain & ((q + magic) - magic == q) & (q <= above) & (q >= below);
        const uint64_t hard = (odd ? ~0ull : __builtin_amdgcn_ballot_w64(!easy)) & (~0ull << from);
        if (hard == 0) return (float)(off + lane_value(upto, 63));
        const uint32_t l = __builtin_ctzll(hard);
        float t = odd & (lane == from) ? s : (float)q;
#pragma unroll
        for (int k = 0; k < 8; k++) t += f[k];
        const uint64_t even = __builtin_amdgcn_ballot_w64(((double)t + grid) - grid == (double)t);
        s = u2f(lane_value(f2u(t), l));
        off = lane_value((double)t - upto, l);
        odd = !((even >> l) & 1);
        from = l + 1;
    }
    return s;
}

// T(x*x)'s (v: the squares, s: the sum's bit pattern).  From approximate sums in front of the lanes every lane takes the binade it adds in; a lane
// is clean if its run starts and ends there, with a margin for what the approximation can be off by.  Pairs of distances as in
// ordered_add; the parity in front of a lane is followed for both parities that its stretch of clean lanes can start with, and the
// distances are summed under both.  Then the lanes that are not clean (about eight of a row, where the sum passes a power of two)
// are taken in order: the stretch in front of one is a single addition, its own run is added for real.  What the approximation claims is checked
// on the exact sum, and a step on which it fails goes through ordered_add.
template <class C>
__device__ __forceinline__ uint32_t norm_ordered_squares(uint32_t s, const v4u& v, uint32_t lane) {
    const uint32_t start = s;
    const float run = u2f(C::one(0, v)), upto = lanes_scan(run), carry = u2f(s);
    const uint32_t e = f2u((carry + upto) * (1.0f + 0x1p-10f)) >> 23;
    const bool clean = (e - 2 < 252) & (f2u((carry + (upto - run)) * (1.0f - 0x1p-10f)) >> 23 == e);
    const uint32_t base = e << 23;
    typename C::Pair p = C::pair(base, base + 1);
    C::run(p, v);
    const uint32_t d0 = clean ? C::lo(p) - base : 0, d1 = clean ? C::hi(p) - (base + 1) : 0;
    const uint64_t dirty = __builtin_amdgcn_ballot_w64(!clean);
    const uint64_t odd = __builtin_amdgcn_ballot_w64(d0 & 1u), tie = __builtin_amdgcn_ballot_w64(d0 != d1);
    const uint32_t flip = __builtin_amdgcn_mbcnt_hi((uint32_t)(odd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odd, 0));
    const uint64_t flips = __builtin_amdgcn_ballot_w64(flip & 1u);
    const uint64_t set = tie | dirty, gen0 = set & flips, gen1 = gen0 ^ dirty;
    const uint64_t prop0 = gen0 | ~set, prop1 = gen1 | ~set;
    const uint32_t u0 = lanes_scan(__builtin_amdgcn_inverse_ballot_w64(((prop0 + gen0) ^ prop0 ^ gen0) ^ flips) ? d1 : d0);
    const uint32_t u1 = lanes_scan(__builtin_amdgcn_inverse_ballot_w64(((prop1 + gen1 + 1) ^ prop1 ^ gen1) ^ flips) ? d1 : d0);
    bool failed = false;
    uint64_t todo = dirty;
    uint32_t from = 0, c0 = 0, c1 = 0;
    for (;;) {
        const uint32_t at = todo ? __builtin_ctzll(todo) : 64, last = at < 64 ? at : 63;             // (a dirty lane's own distance is zero)
        const uint32_t n0 = lane_value(u0, last), n1 = lane_value(u1, last), eb = lane_value(base, at ? at - 1 : 0);
        if (at > from) {
            failed |= (s ^ eb) >> 23 != 0;
            s += s & 1u ? n1 - c1 : n0 - c0;
            failed |= (s ^ eb) >> 23 != 0;
        }
        if (at == 64) break;
        s = lane_value(C::one(s, v), at);
        c0 = n0;
        c1 = n1;
        from = at + 1;
        todo &= todo - 1;
    }
    if (failed) {
        const v4u one[1] = {v};
        s = ordered_add<C, 1, 3>(start, one, lane);
    }
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
            if (KIND == NORM_LAYER && (open & 2)) s1 = norm_ordered_sum<T>(s1, here, lane);
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
    RT_REQUIRE(rows <= 0x7fffffffull, RT_ERR_SIZE, "norm: too many rows");
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
    return bf16 ? launch_norm16_row<bf16_t, NORM_RMS>(dev, x, scale, bias, y, rows, cols, eps)
                : launch_norm16_row<half_t, NORM_RMS>(dev, x, scale, bias, y, rows, cols, eps);
}
