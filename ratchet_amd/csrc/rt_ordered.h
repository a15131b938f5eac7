// Left-to-right floating-point sums of a row, reproduced bit for bit by a whole wave without walking the row.
//
// The reference adds the terms of a row one by one, s <- fl(s + a), and the rounding of every add depends on the running sum.  What
// makes the chain divisible: while s stays inside one binade, [2^e, 2^(e+1)), it is 2^e + k * ulp with an integer k, and what the add
// of a term a >= 0 does to k depends on s only through the parity of k (round to nearest even: the parity decides ties).  A run
// of adds that stays inside the binade is therefore a function k -> k + d[k & 1] of two constants.  Both come out of the adder
// itself: the run is added up twice, from 2^e and from 2^e + ulp, and d[p] is the distance the p-th sum has moved, read off the bit
// patterns.  d[0] == d[1] when no tie occurred (both sums moved alike); otherwise both ended on the same parity, whatever they started from.
//
// ordered_add takes one run per lane.  Every lane adds its run up from the binade the sum is in at the moment; the parity at the start
// of each lane's run follows from the lanes before it by one 64-bit addition on the scalar unit (a lane with a tie sets the
// parity, the others flip or keep it: generate, kill and propagate of a carry chain); the chosen distances are summed over the
// lanes.  If the sum leaves the binade in a lane, that lane's run is added for real to the exact sum before it, in the same pass that
// prepares the lanes behind it for the next binade: a pass for every binade the sum passes through, and one for every run of 64.
// Nothing is approximated: a result is used only if the sum stayed inside the binade it was made for (the sum never
// decreases, so every sum in between did too).  inf and NaN lie beyond every binade and are absorbed as the adder absorbs them.
#ifndef RT_ORDERED_H
#define RT_ORDERED_H

#include "rt_arith.h"
#include "rt_internal.h"

namespace {

// inclusive prefix sum over the 64 lanes, by DPP moves inside rows of 16 and from row to row
template <int CTRL, int ROWS> __device__ __forceinline__ uint32_t scan_move(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ uint32_t lanes_scan(uint32_t v) {
    v += scan_move<0x111, 0xf>(v);                           // row_shr:1, 2, 4, 8
    v += scan_move<0x112, 0xf>(v);
    v += scan_move<0x114, 0xf>(v);
    v += scan_move<0x118, 0xf>(v);
    v += scan_move<0x142, 0xa>(v);                           // the last lane of rows 0 and 2 onto rows 1 and 3
    v += scan_move<0x143, 0xc>(v);                           // lane 31 onto lanes 32 .. 63
    return v;
}
__device__ __forceinline__ float lanes_scan(float v) {
#define RT_SCAN_STEP(C, R) v += u2f(scan_move<C, R>(f2u(v)))
    RT_SCAN_STEP(0x111, 0xf);
    RT_SCAN_STEP(0x112, 0xf);
    RT_SCAN_STEP(0x114, 0xf);
    RT_SCAN_STEP(0x118, 0xf);
    RT_SCAN_STEP(0x142, 0xa);
    RT_SCAN_STEP(0x143, 0xc);
#undef RT_SCAN_STEP
    return v;
}
__device__ __forceinline__ double lanes_scan(double v) {
#define RT_SCAN_STEP(C, R)                                                                                              \
    do {                                                                                                                \
        const uint64_t u = __builtin_bit_cast(uint64_t, v);                                                             \
        const uint64_t o = (uint64_t)scan_move<C, R>((uint32_t)(u >> 32)) << 32 | scan_move<C, R>((uint32_t)u);         \
        v += __builtin_bit_cast(double, o);                                                                             \
    } while (0)
    RT_SCAN_STEP(0x111, 0xf);
    RT_SCAN_STEP(0x112, 0xf);
    RT_SCAN_STEP(0x114, 0xf);
    RT_SCAN_STEP(0x118, 0xf);
    RT_SCAN_STEP(0x142, 0xa);
    RT_SCAN_STEP(0x143, 0xc);
#undef RT_SCAN_STEP
    return v;
}
// lane i - 1's value, zero in lane 0
__device__ __forceinline__ float lane_before(float v) { return u2f(scan_move<0x138, 0xf>(f2u(v))); }

__device__ __forceinline__ uint32_t lane_value(uint32_t v, uint32_t lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ double lane_value(double v, uint32_t lane) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    return __builtin_bit_cast(double, (uint64_t)lane_value((uint32_t)(u >> 32), lane) << 32 | lane_value((uint32_t)u, lane));
}

// The f32 chain of 16-bit terms.  MANT: mantissa bits of the running sum's type, INF: its infinity's bit pattern.  pair(a, b) starts two sums at two bit
// patterns, run() adds a vector's eight terms to both, lo() and hi() are the sums' bit patterns; one() adds to a single sum.
template <typename T> struct ChainF32;
template <> struct ChainF32<half_t> {
    static constexpr int MANT = 23;
    static constexpr uint32_t INF = 0x7f800000u;
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
    static constexpr int MANT = 23;
    static constexpr uint32_t INF = 0x7f800000u;
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

// s, the same in all lanes: the bit pattern of a running sum of terms >= 0 (or NaN).  Returns that of the sum after the 64 runs of NV
// vectors, lane 0's first.  At the start of a row, where the sum doubles every few lanes, SERIAL lanes are added one by one.
template <class C, int NV, int SERIAL>
__device__ __forceinline__ uint32_t ordered_add(uint32_t s, const v4u (&v)[NV], uint32_t lane) {
    constexpr uint32_t ULPS = 1u << C::MANT;                 // sums in a binade
    uint32_t from = 0;                                       // lanes below it are in s
    if (s == 0) {
        for (; from < SERIAL; from++) {
            uint32_t t = s;
#pragma unroll
            for (int k = 0; k < NV; k++) t = C::one(t, v[k]);
            s = lane_value(t, from);
        }
    }
    bool real = false;                                       // lane `from` adds to s itself
    uint32_t e = s >> C::MANT;
    while (s < C::INF) {
        // the binade; the subnormals and the first normal one have one ulp and count as one
        const uint32_t base = e <= 1 ? 0 : e << C::MANT, size = e <= 1 ? 2 * ULPS : ULPS;
        const bool mine = real && lane == from;
        typename C::Pair p = C::pair(mine ? s : base, base + 1);
#pragma unroll
        for (int k = 0; k < NV; k++) C::run(p, v[k]);
        uint32_t d0 = C::lo(p) - base, d1 = C::hi(p) - (base + 1);
        if (real) {
            s = lane_value(C::lo(p), from);
            if (++from == 64) return s;
            real = false;
            if (s >> C::MANT != e && !(e <= 1 && s >> C::MANT <= 1)) {       // not in the binade that the lanes behind prepared for
                e = s >> C::MANT;
                continue;
            }
        }
        if (C::MANT == 23) {                                 // (64 distances have to fit into a word)
            d0 = d0 < 2 * ULPS ? d0 : 2 * ULPS;
            d1 = d1 < 2 * ULPS ? d1 : 2 * ULPS;
        }
        if (lane < from) d0 = d1 = 0;
        // the parity in front of each lane: `flips` is that of the distances before it alone, a tie in between sets it anew
        const uint64_t odd = __builtin_amdgcn_ballot_w64(d0 & 1u), tie = __builtin_amdgcn_ballot_w64(d0 != d1);
        const uint32_t below = __builtin_amdgcn_mbcnt_hi((uint32_t)(odd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odd, 0));
        const uint64_t flips = __builtin_amdgcn_ballot_w64(below & 1u);
        const uint64_t gen = tie & flips, prop = gen | ~tie;
        const uint64_t parity = ((prop + gen + (s & 1u)) ^ prop ^ gen) ^ flips;
        const uint32_t d = __builtin_amdgcn_inverse_ballot_w64(parity) ? d1 : d0;
        const uint32_t upto = lanes_scan(d);
        const uint64_t leaves = __builtin_amdgcn_ballot_w64(upto >= base + size - s);
        if (leaves == 0) return s + lane_value(upto, 63);
        const uint32_t at = __builtin_ctzll(leaves);
        s += lane_value(upto, at) - lane_value(d, at);
        from = at;
        real = true;
        e = e <= 1 ? 2 : e + 1;                              // where the lanes behind that one most likely add
    }
    // inf or NaN: the next lane that makes anything else of it makes a NaN, which stays
    uint32_t t = s;
#pragma unroll
    for (int k = 0; k < NV; k++) t = C::one(t, v[k]);
    const uint64_t other = __builtin_amdgcn_ballot_w64(lane >= from && t != s);
    return other ? lane_value(t, __builtin_ctzll(other)) : s;
}

}  // namespace

#endif
