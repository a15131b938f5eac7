// Left-to-right floating-point sums of a row, reproduced bit for bit by a whole wave without walking the row.
//
// The reference adds the terms of a row one by one, s <- fl(s + a), and the rounding of every add depends on the running sum.  What
// makes the chain divisible: while s stays inside one binade, [2^e, 2^(e+1)), it is 2^e + k * ulp with an integer k, and what the add
// of a term a >= 0 does to k depends on s only through the parity of k (round to nearest even: the parity decides ties).  A run
// of adds that stays inside the binade is therefore a function k -> k + d[k & 1] of two constants.  Both come out of the adder
// itself: the run is added up twice, from 2^e and from 2^e + ulp, and d[p] is the distance the p-th sum has moved, read off the bit
// patterns.  d[0] == d[1] when no tie occurred (both sums moved alike); otherwise both ended on the same parity, whatever they started from.
//
// One run per lane: every lane adds its run up from the binade that the sum is in there; the parity at the start of each lane's run follows from the
// lanes before it by one 64-bit addition on the scalar unit (a lane with a tie sets the parity, the others flip or keep it: generate, kill and
// propagate of a carry chain); the chosen distances are summed over the lanes.  Lanes in which the sum leaves the binade add for real to the exact sum before them.
// norm_ordered_squares below and sr_group_add (rt_softmax_row.hip) do that, each where its sums need it.
#ifndef RT_ORDERED_H
#define RT_ORDERED_H

#include <cmath>
#include <cstdint>

// (v4u, u2f, f2u and wave_max come from the includer, rt_arith.h on the GPU: the text is compiled for the host as well, where
// tests/ordered_sums_check.cpp compares the 64 lanes' sums with the plain ones)
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

// the ulp of the binade of m (m finite, at least 2^-103; zero below that)
__device__ __forceinline__ float nr_ulp(float m) {
    const uint32_t e = f2u(m) >> 23;
    return e > 23 ? u2f((e - 23) << 23) : 0.0f;
}
// what f, a value of a 16-bit type, is off the nearest multiple of u = magic * 2^-23 / 1.5, a power of two or zero: zero, or NaN for inf and
// NaN, if it is none.  (Up to 2^22 u the sum has the ulp u; values beyond 2^11 u have no bit below u.)
__device__ __forceinline__ float nr_off(float f, float magic) {
    return f - ((f + magic) - magic);
}

// Both ordered sums take a step of 512 columns, 64 vectors, one a lane.
//
// x's: up to a lane the sum runs exactly, and is q (in double), as long as the lanes before it are `easy`: their terms and their q are
// multiples of the ulp of the binade that their partial sums stay in.  A lane's own sums, added up from zero, can reach twice as far as the
// running sum does (from -0.9 to 0.9 of the binade, say) and must not round on the way: in f32 they may from 2^24 ulp on, and then all lanes add
// theirs up again in double.  (Such lanes are one or two in a step of a sum that crosses zero.  Adding for real in each of them cost more:
// bf16 LayerNorm [1024,2560] of rows without a mean 13.0 us, 11.2 so.)  The first lane that is not easy adds its eight terms to the exact sum
// for real, and the lanes behind it start from there.
// N::widen(x, f): a vector's eight values as floats.
template <class N>
__device__ __forceinline__ float norm_ordered_sum(float s, const v4u& x, uint32_t lane) {
    float f[8], part = 0.0f, low = 0.0f, high = 0.0f;        // a lane's sum, the ends of its partial sums
    N::widen(x, f);
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
    // (a sum of 2^24 ulp may have been rounded to that, one of less has not been)
    double own = (double)part, least = (double)low, most = (double)high;
    const float exact = ulp * 0x1p24f;
    if (__builtin_amdgcn_ballot_w64(plain & ((high >= exact) | (low <= -exact)))) {
        own = least = most = 0.0;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            own += (double)f[k];
            least = __builtin_fmin(least, own);
            most = __builtin_fmax(most, own);
        }
    }
    // no terms but zeros: nothing to add, whatever the sum is (past the row's end, where a sum that has cancelled is below every ulp above, each such
    // lane took a turn of its own)
    const bool none = ((x[0] | x[1] | x[2] | x[3]) & 0x7fff7fffu) == 0;
    const double mine = plain ? own : 0.0, upto = lanes_scan(mine), before = upto - mine;
    const double limit = (double)ulp * 0x1p24, magic = (double)ulp * 0x1.8p52;       // sums up to the limit in steps of ulp are f32 values
    const double above = limit - most, below = -limit - least;
    // multiples of coarse * 2^-20, like the lanes' sums, each of which is below 2^26 coarse: so is what is added up from them below 2^33 coarse, and exact
    const double grid = (double)coarse * 0x1.8p32;
    double off = (double)s;                                  // the running sum less `before`, or, odd, what a double cannot hold:
    bool odd = !((off + grid) - grid == off);                // then the next lane adds to s itself
    for (uint32_t from = 0; from < 64;) {
        const double q = off + before;
        const bool easy = none | (plain & ((q + magic) - magic == q) & (q <= above) & (q >= below));
        const uint64_t hard = (odd ? ~0ull : __builtin_amdgcn_ballot_w64(!easy)) & (~0ull << from);
        if (hard == 0) return (float)(off + lane_value(upto, 63));
        const uint32_t l = __builtin_ctzll(hard);
        float t = (odd & (lane == from)) ? s : (float)q;
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
// is clean if its run starts and ends there, with a margin for what the approximation can be off by: the margin is 2^-10, and the approximate and the ordered
// sum, each of 512 terms >= 0 on the same exact sum, are off the true one by 2^-15 at most, in a clean lane of the binade that both ends lie in (a term so
// large that what it hides matters takes its lane out of the binade).  So is the binade right for a stretch of clean lanes, which all have the same.  Pairs of
// distances as above; the parity in front of a lane is followed for both parities that its stretch of clean lanes can start with, and the
// distances are summed under both.  Then the lanes that are not clean (about eight of a row, where the sum passes a power of two; all where it is
// subnormal, near overflow or NaN) are taken in order: the stretch in front of one is a single addition, its own run is added for real.  A lane without terms, past
// the row's end, has no distance whatever the sum is: of a sum within the margin of a power of two each took a turn (f16 RMSNorm [667,2056] 11.6 us, 6.5 so).
template <class C>
__device__ __forceinline__ uint32_t norm_ordered_squares(uint32_t s, const v4u& v, uint32_t lane) {
    const float run = u2f(C::one(0, v)), upto = lanes_scan(run), carry = u2f(s);
    const uint32_t e = f2u((carry + upto) * (1.0f + 0x1p-10f)) >> 23;
    const bool clean = (e - 2 < 252) & (f2u((carry + (upto - run)) * (1.0f - 0x1p-10f)) >> 23 == e);
    const uint32_t base = e << 23;
    typename C::Pair p = C::pair(base, base + 1);
    C::run(p, v);
    const uint32_t d0 = clean ? C::lo(p) - base : 0, d1 = clean ? C::hi(p) - (base + 1) : 0;
    // (no terms but zeros: nothing to add, whatever the sum is)
    const uint64_t dirty = __builtin_amdgcn_ballot_w64(!clean & ((v[0] | v[1] | v[2] | v[3]) != 0));
    const uint64_t odd = __builtin_amdgcn_ballot_w64(d0 & 1u), tie = __builtin_amdgcn_ballot_w64(d0 != d1);
    const uint32_t flip = __builtin_amdgcn_mbcnt_hi((uint32_t)(odd >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)odd, 0));
    const uint64_t flips = __builtin_amdgcn_ballot_w64(flip & 1u);
    const uint64_t set = tie | dirty, gen0 = set & flips, gen1 = gen0 ^ dirty;
    const uint64_t prop0 = gen0 | ~set, prop1 = gen1 | ~set;
    const uint32_t u0 = lanes_scan(__builtin_amdgcn_inverse_ballot_w64(((prop0 + gen0) ^ prop0 ^ gen0) ^ flips) ? d1 : d0);
    const uint32_t u1 = lanes_scan(__builtin_amdgcn_inverse_ballot_w64(((prop1 + gen1 + 1) ^ prop1 ^ gen1) ^ flips) ? d1 : d0);
    uint64_t todo = dirty;
    uint32_t from = 0, c0 = 0, c1 = 0;
    for (;;) {
        const uint32_t at = todo ? __builtin_ctzll(todo) : 64, last = at < 64 ? at : 63;             // (a dirty lane's own distance is zero)
        const uint32_t n0 = lane_value(u0, last), n1 = lane_value(u1, last);
        if (at > from) s += s & 1u ? n1 - c1 : n0 - c0;
        if (at == 64) return s;
        s = lane_value(C::one(s, v), at);
        c0 = n0;
        c1 = n1;
        from = at + 1;
        todo &= todo - 1;
    }
}

}  // namespace

#endif
