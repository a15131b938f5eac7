// Host check of the wave-per-row norms' ordered sums (ratchet_amd/csrc/rt_ordered.h, the kernel's own text) against the plain
// left-to-right f32 sum.  The 64 lanes are 64 contexts that run in turn from one exchange between lanes to the next.
// Rows: N(0, 1); with an offset; spread magnitudes; values and their negatives shuffled, which cancel to zero after large excursions; runs that
// swing between signs inside and between the lanes, by up to 2^24 of their last bits; tiny and huge ones; inf and NaN; the rows of
// `found`.  Sums go on over the steps of a row, from the plain sum of the steps before.
// Build: g++ -O2 -std=c++17 -ffp-contract=off -I ratchet_amd/csrc.   Usage: ordered_sums_check ROWS
// prints "sum_f16 <n> sum_bf16 <n> squares_f16 <n> squares_bf16 <n> turns <k> centred <c> checked <m>" (n: steps whose sums differ; k: the most exchanges
// between lanes in a step whose upper lanes have no terms, of rows that cancel and of squares next to a power of two; c: the mean of them in steps of rows without a mean), exit code 0 iff
// all n are 0, k is at most MOST_TURNS and c at most MEAN_TURNS.
#include <ucontext.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include <cstdint>

typedef uint32_t v4u __attribute__((vector_size(16)));
static inline float u2f(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static inline uint32_t f2u(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }

// ---- a wave of 64 contexts
static const int LANES = 64;
static ucontext_t home, at[LANES];
static std::vector<char> stacks(LANES * 65536);
static int me;
static uint64_t slot[2][LANES];
static unsigned turn[LANES];
static void (*work)(int);

// every lane leaves a value; once all have, each goes on with all of them
static const uint64_t* exchange(uint64_t v) {
    const int self = me;
    uint64_t* const s = slot[turn[self]++ & 1];
    s[self] = v;
    me = (self + 1) % LANES;
    swapcontext(&at[self], &at[me]);
    return s;
}
static void lane_main() {
    const int self = me;
    work(self);
    if (self == LANES - 1) setcontext(&home);                // the last one to end: all lanes make the same exchanges
    me = self + 1;
    setcontext(&at[me]);
}
static void run_wave(void (*f)(int)) {
    work = f;
    for (int i = 0; i < LANES; i++) {
        getcontext(&at[i]);
        at[i].uc_stack.ss_sp = &stacks[i * 65536];
        at[i].uc_stack.ss_size = 65536;
        at[i].uc_link = nullptr;
        makecontext(&at[i], lane_main, 0);
        turn[i] = 0;
    }
    me = 0;
    swapcontext(&home, &at[0]);
}

// ---- the operations between lanes that the text uses
static inline uint64_t __builtin_amdgcn_ballot_w64(bool b) {
    const uint64_t* s = exchange(b);
    uint64_t m = 0;
    for (int i = 0; i < LANES; i++) m |= s[i] << i;
    return m;
}
static inline bool __builtin_amdgcn_inverse_ballot_w64(uint64_t m) { return m >> me & 1; }
static inline uint32_t __builtin_amdgcn_mbcnt_lo(uint32_t m, uint32_t n) {
    return n + (uint32_t)__builtin_popcountll((uint64_t)m & ((1ull << me) - 1));
}
static inline uint32_t __builtin_amdgcn_mbcnt_hi(uint32_t m, uint32_t n) {
    return n + (uint32_t)__builtin_popcountll((uint64_t)m << 32 & ((1ull << me) - 1));
}
static inline uint32_t __builtin_amdgcn_readlane(uint32_t v, uint32_t lane) { return (uint32_t)exchange(v)[lane]; }
static inline uint32_t __builtin_amdgcn_readfirstlane(uint32_t v) { return (uint32_t)exchange(v)[0]; }
// the moves of the scans: within rows of 16 by 1, 2, 4, 8 lanes; the last lane of a row, or lane 31, onto what follows; the whole wave by one
static inline int __builtin_amdgcn_update_dpp(int old, int v, int ctrl, int rows, int, bool) {
    const uint64_t* s = exchange((uint32_t)v);
    if (!(rows >> (me / 16) & 1)) return old;
    int from = -1;
    if (ctrl > 0x110 && ctrl < 0x120) from = me % 16 >= (ctrl & 15) ? me - (ctrl & 15) : -1;
    else if (ctrl == 0x138) from = me - 1;
    else if (ctrl == 0x142) from = me / 16 * 16 - 1;
    else if (ctrl == 0x143) from = me >= 32 ? 31 : -1;
    else abort();
    return from < 0 ? old : (int)(uint32_t)s[from];
}
static inline float wave_max(float v) {
    const uint64_t* s = exchange(f2u(v));
    float m = u2f((uint32_t)s[0]);
    for (int i = 1; i < LANES; i++) m = __builtin_fmaxf(m, u2f((uint32_t)s[i]));
    return m;
}

#define __device__
#define __forceinline__ inline
#pragma GCC diagnostic ignored "-Wunknown-pragmas"
#include "rt_ordered.h"

// ---- the 16-bit types
static float from_f16(uint16_t h) {
    const uint32_t m = h & 0x7fff, sign = (uint32_t)(h & 0x8000) << 16;
    if (m >= 0x7c00) return u2f(sign | 0x7f800000u | (m & 0x3ff) << 13);
    const float f = m & 0x7c00 ? u2f((m << 13) + 0x38000000u) : (float)m * 0x1p-24f;
    return u2f(f2u(f) | sign);
}
static uint16_t to_f16(float f) {                            // nearest even
    const uint16_t sign = (uint16_t)(f2u(f) >> 16 & 0x8000);
    f = fabsf(f);
    if (f != f) return 0x7e00;
    if (f >= 65520.0f) return sign | 0x7c00;
    if (f < 0x1p-14f) return sign | (uint16_t)(f2u(f + 0.5f) - 0x3f000000u);
    const uint32_t u = f2u(f);
    return sign | (uint16_t)((u + 0xfffu + ((u >> 13) & 1u) - 0x38000000u) >> 13);
}
static float from_bf16(uint16_t h) { return u2f((uint32_t)h << 16); }
static uint16_t to_bf16(float f) {
    const uint32_t u = f2u(f);
    if (f != f) return 0x7fc0;
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
template <bool BF> struct Half {
    static float widen(uint16_t h) { return BF ? from_bf16(h) : from_f16(h); }
    static uint16_t round(float f) { return BF ? to_bf16(f) : to_f16(f); }
    static void widen(const v4u& x, float (&f)[8]) {
        for (int q = 0; q < 8; q++) f[q] = widen((uint16_t)(x[q / 2] >> 16 * (q & 1)));
    }
    // the chain of norm_ordered_squares
    struct Pair { float a, b; };
    static Pair pair(uint32_t a, uint32_t b) { return Pair{u2f(a), u2f(b)}; }
    static uint32_t lo(const Pair& p) { return f2u(p.a); }
    static uint32_t hi(const Pair& p) { return f2u(p.b); }
    static void run(Pair& p, const v4u& v) {
        float f[8];
        widen(v, f);
        for (float t : f) { p.a += t; p.b += t; }
    }
    static uint32_t one(uint32_t s, const v4u& v) {
        float f[8], a = u2f(s);
        widen(v, f);
        for (float t : f) a += t;
        return f2u(a);
    }
};

static const uint16_t* terms;                                // the 512 of the step
static float s_in, s_out[LANES];
template <bool BF, bool SQUARES> static void lane_work(int lane) {
    v4u v;
    memcpy(&v, terms + lane * 8, 16);
    s_out[lane] = SQUARES ? u2f(norm_ordered_squares<Half<BF>>(f2u(s_in), v, (uint32_t)lane)) : norm_ordered_sum<Half<BF>>(s_in, v, (uint32_t)lane);
}
static unsigned long long checked;
template <bool BF, bool SQUARES> static unsigned long long differ(const std::vector<float>& row) {
    std::vector<uint16_t> t(row.size());
    for (size_t i = 0; i < row.size(); i++) {
        t[i] = Half<BF>::round(row[i]);
        if (SQUARES) t[i] = Half<BF>::round(Half<BF>::widen(t[i]) * Half<BF>::widen(t[i]));
    }
    unsigned long long bad = 0;
    float s = 0.0f;
    for (size_t i = 0; i < t.size(); i += 512) {
        float want = s;
        for (int k = 0; k < 512; k++) want += Half<BF>::widen(t[i + k]);
        terms = &t[i];
        s_in = s;
        run_wave(lane_work<BF, SQUARES>);
        bool same = true;
        for (float got : s_out) same &= want != want ? got != got : f2u(got) == f2u(want);
        bad += !same;
        checked++;
        s = want;
    }
    return bad;
}

int main(int argc, char** argv) {
    const int rows = argc > 1 ? atoi(argv[1]) : 100;
    std::mt19937_64 rng(7);
    std::normal_distribution<float> normal;
    auto below = [&](int n) { return (int)(rng() % (uint64_t)n); };
    std::vector<std::vector<float>> found;
    {
        std::vector<float> r(512, 0.0f);                     // lane 1's own sum rounds, the running one does not
        r[0] = -127; r[8] = 100; r[9] = 50; r[10] = 0x1p-17f; r[16] = 0x1p-7f;
        found.push_back(r);
        r.assign(512, 0.0f);                                 // the same in bf16 values
        std::fill(r.begin(), r.begin() + 5, -3063808.0f);
        r[8] = 1;
        std::fill(r.begin() + 9, r.begin() + 16, 3506176.0f);
        r[16] = -9240576; r[17] = 16384;
        found.push_back(r);
        r.assign(512, 0.0f);                                 // a lane whose sum of 2^24 + 1 ulps rounds to 2^24
        r[0] = -5; r[8] = 4; r[9] = 4; r[10] = 0x1p-21f; r[16] = 0x1p-7f;
        found.push_back(r);
        for (size_t k = 0, n = found.size(); k < n; k++) {
            r = found[k];
            for (float& f : r) f = -f;
            found.push_back(r);
        }
    }
    unsigned long long bad[4] = {0, 0, 0, 0};
    for (int n = 0; n < rows + (int)found.size(); n++) {
        std::vector<float> r(n < (int)found.size() ? 512 : 512 * (1 + below(5)));
        if (n < (int)found.size()) {
            r = found[n];
        } else {
            const int kind = n % 9;
            const float scale = std::exp2((float)(below(24) - 12));
            for (size_t i = 0; i < r.size(); i++) {
                const float f = normal(rng);
                switch (kind) {
                    case 0: case 4: r[i] = f; break;
                    case 1: r[i] = 3.0f + 0.1f * f; break;
                    case 2: r[i] = f * std::exp2(-(float)below(18)); break;
                    case 3: r[i] = f * f * f * scale; break;
                    case 5: case 6: r[i] = (i / (kind == 5 ? 8 : 4 + below(9)) % 2 ? 20.0f : -20.0f) * scale * (1.0f + 0.3f * f) * (below(4) ? 1.0f : std::exp2(-(float)below(24))); break;
                    case 7: r[i] = f * (below(2) ? 0x1p-14f : 0x1p-24f); break;
                    default: r[i] = f * (below(2) ? 0x1p12f : 0x1p14f); break;
                }
            }
            if (kind == 4 || kind == 2 || (kind == 3 && below(2))) {         // values and their negatives
                for (size_t i = 1; i < r.size(); i += 2) r[i] = -r[i - 1];
                std::shuffle(r.begin(), r.end(), rng);
            }
            if (below(12) == 0) r[below((int)r.size())] = below(3) ? INFINITY : NAN;
            if (below(12) == 0) r[below((int)r.size())] = -INFINITY;
        }
        bad[0] += differ<false, false>(r);
        bad[1] += differ<true, false>(r);
        bad[2] += differ<false, true>(r);
        if (n % 9 == 7 || n % 9 == 8) for (float& f : r) f *= n % 9 == 7 ? 0x1p-50f : 0x1p46f;        // (squares at the ends of bf16)
        bad[3] += differ<true, true>(r);
    }
    // 40 exchanges for the scans and votes of a step and five for each lane that adds for real: a few, not all that have no terms
    const unsigned MOST_TURNS = 40 + 5 * 12;
    unsigned turns = 0;
    for (int n = 0; n < 40; n++) {
        std::vector<float> r(512, 0.0f);
        const int cols = 8 * (2 + below(40));
        for (int i = 0; i < cols; i += 2) r[i + 1] = -(r[i] = normal(rng));
        std::shuffle(r.begin(), r.begin() + cols, rng);
        bad[0] += differ<false, false>(r);
        turns = std::max(turns, turn[0]);
        bad[1] += differ<true, false>(r);
        turns = std::max(turns, turn[0]);
    }
    // the squares of rows whose sum ends next to a power of two, with few terms in their last step
    for (int n = 0; n < 40; n++) {
        std::vector<float> r(1024, 0.0f);
        double total = 0;
        const int cols = 512 + 8 * (1 + below(20));
        for (int i = 0; i < cols; i++) total += (r[i] = normal(rng)) * (double)r[i];
        const float by = (float)std::sqrt(std::exp2(below(16) - 4) / total);
        for (int i = 0; i < cols; i++) r[i] *= by;
        bad[2] += differ<false, true>(r);
        turns = std::max(turns, turn[0]);
        bad[3] += differ<true, true>(r);
        turns = std::max(turns, turn[0]);
    }
    // 25 exchanges for the scans and votes of a step; a lane adds for real in fewer than half of the steps (each in which the lane's own sum passes 2^24
    // of its last bits, where the running one crosses zero, would make it 33 on average)
    const double MEAN_TURNS = 30;
    unsigned long long exchanges = 0, steps = 0;
    for (int n = 0; n < 40; n++) {
        std::vector<float> r(5 * 512);
        double mean = 0;
        for (float& f : r) mean += (f = normal(rng)) / (double)r.size();
        for (float& f : r) f -= (float)mean;
        for (bool bf : {false, true}) {
            float s = 0.0f;
            for (size_t i = 0; i < r.size(); i += 512, steps++) {
                uint16_t t[512];
                float want = s;
                for (int k = 0; k < 512; k++) {
                    t[k] = bf ? to_bf16(r[i + k]) : to_f16(r[i + k]);
                    want += bf ? from_bf16(t[k]) : from_f16(t[k]);
                }
                terms = t;
                s_in = s;
                run_wave(bf ? lane_work<true, false> : lane_work<false, false>);
                for (float got : s_out) bad[bf] += f2u(got) != f2u(want);
                exchanges += turn[0];
                s = want;
            }
        }
    }
    const double centred = (double)exchanges / (double)steps;
    printf("sum_f16 %llu sum_bf16 %llu squares_f16 %llu squares_bf16 %llu turns %u centred %.1f checked %llu\n", bad[0], bad[1], bad[2], bad[3], turns, centred,
           checked);
    return bad[0] || bad[1] || bad[2] || bad[3] || turns > MOST_TURNS || centred > MEAN_TURNS;
}
