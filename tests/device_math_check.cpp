// Host check of the kernels' libm-level routines: ratchet_amd/csrc/rt_libm.h compiled as plain C++ against this machine's
// C library, which is what the reference's f32::tanh / f32::exp / f32::ln / f32::sin / f32::cos resolve to
// (crates/ratchet-core/src/cpu/unary.rs:46-65, cpu/softmax.rs:30).  Bit equality is required (any NaN equals any NaN).
// Inputs: every `stride`-th float bit pattern over the whole 2^32 range (stride 1 = exhaustive), every value that a 16-bit
// input can widen to, and the breakpoints of the algorithms.  Build: g++ -O2 -ffp-contract=off.
// Usage: device_math_check [stride]   -> prints "tanhf <n> expm1f <n> expf <n> logf <n> sinf <n> cosf <n> f2bf <n> checked <m>", exit code 0 iff all n are 0.
//
// The kernels compile the same text but for two expressions of rt_tanhf that rt_math.h replaces: the median of three by the
// instruction for it, which gives the same values, and the division by rt_div_mid, which is not correctly rounded for all
// operands and whose result may hang on the last bit of the GPU's reciprocal instruction.  What that can change is found
// here: the short division with each reciprocal correctly rounded, an ulp lower and an ulp higher (the instruction is
// within one), in all combinations.  With correctly rounded reciprocals every result is the C library's; with the others
// 113 positive inputs (and their negatives) differ, which tests/golden/tanh_division_inputs.txt lists and
// test_tanh_where_the_division_hangs_on_the_reciprocal puts to the GPU.  All other inputs give the C library's result
// whichever of the three the instruction returns.
// Usage: device_math_check division FILE [stride]   -> every `stride`-th positive float: prints the sensitive inputs that
//   FILE does not list, then "sensitive <n> unlisted <n> listed <n> insensitive <n> wrong <n> checked <m>" (insensitive: of the
//   listed; wrong: with correctly rounded reciprocals); exit code 0 iff unlisted, insensitive and wrong are 0.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>

// 0: the plain division; 1: rt_div_mid of rt_math.h, its reciprocals off by off[0] and off[1] ulps
static int division = 0, off[2], nth;
static inline float divide(float n, float d) {
    if (division == 0) return n / d;
    float r = 1.0f / d;
    uint32_t bits;
    memcpy(&bits, &r, 4);
    bits += (uint32_t)off[nth++ & 1];
    memcpy(&r, &bits, 4);
    const float q = n * r;
    return fmaf(fmaf(-d, q, n), r, q);
}
#define RT_DIV(n, d) divide(n, d)
#define RT_FN static inline
#define RT_TABLE static const
#include "rt_libm.h"

static inline bool same(float a, float b) { return f2u(a) == f2u(b) || (a != a && b != b); }

// round to nearest even, NaN quieted with the payload's top bits kept: half::bf16::from_f32
static inline uint16_t bf16_reference(float f) {
    const uint32_t x = f2u(f);
    if ((x & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((x >> 16) | 0x0040u);
    const uint32_t lower = x & 0xffffu, keep = x >> 16;
    if (lower > 0x8000u || (lower == 0x8000u && (keep & 1u))) return (uint16_t)(keep + 1);
    return (uint16_t)keep;
}

struct Counts {
    unsigned long long tanh_bad = 0, expm1_bad = 0, exp_bad = 0, log_bad = 0, sin_bad = 0, cos_bad = 0, bf_bad = 0, checked = 0;
    void one(uint32_t bits) {
        const float x = u2f(bits);
        if (!same(rt_tanhf(x), tanhf(x))) tanh_bad++;
        if (!same(rt_expm1f(x), expm1f(x))) expm1_bad++;
        if (!same(rt_expf(x), expf(x))) exp_bad++;
        if (!same(rt_logf(x), logf(x))) log_bad++;
        if (!same(rt_sinf(x), sinf(x))) sin_bad++;
        if (!same(rt_cosf(x), cosf(x))) cos_bad++;
        if (f2bf(x) != bf16_reference(x)) bf_bad++;
        checked++;
    }
};

static int check_division(const char* file, unsigned long long stride) {
    std::set<uint32_t> listed;
    FILE* f = fopen(file, "r");
    if (!f) return 2;
    char word[256];
    while (fscanf(f, "%255s", word) == 1) {
        if (word[0] == '#') {
            if (!fgets(word, sizeof word, f)) break;                             // a comment's rest
            continue;
        }
        listed.insert((uint32_t)strtoul(word, nullptr, 16));
    }
    fclose(f);
    unsigned long long sensitive = 0, unlisted = 0, insensitive = 0, wrong = 0, checked = 0;
    division = 1;
    auto is_sensitive = [&](uint32_t bits) {
        const float x = u2f(bits), want = tanhf(x);
        bool any = false;
        for (int k = 0; k < 9; k++) {
            off[0] = k / 3 - 1, off[1] = k % 3 - 1, nth = 0;
            const bool differs = !same(rt_tanhf(x), want);
            any |= differs;
            if (k == 4 && differs) wrong++;
        }
        checked++;
        return any;
    };
    for (unsigned long long u = 0; u <= 0x7f800000u; u += stride)
        if (is_sensitive((uint32_t)u)) {
            sensitive++;
            if (!listed.count((uint32_t)u)) unlisted++, printf("%08x\n", (uint32_t)u);
        }
    for (uint32_t u : listed) insensitive += !is_sensitive(u);
    printf("sensitive %llu unlisted %llu listed %llu insensitive %llu wrong %llu checked %llu\n", sensitive, unlisted, (unsigned long long)listed.size(),
           insensitive, wrong, checked);
    return (unlisted | insensitive | wrong) ? 1 : 0;
}

int main(int argc, char** argv) {
    if (argc > 2 && !strcmp(argv[1], "division")) return check_division(argv[2], argc > 3 ? strtoull(argv[3], nullptr, 10) : 1021);
    const unsigned long long stride = argc > 1 ? strtoull(argv[1], nullptr, 10) : 1021;
    Counts c;
    for (unsigned long long u = 0; u < (1ull << 32); u += stride) c.one((uint32_t)u);
    // everything an f16 or bf16 input widens to
    for (uint32_t h = 0; h < 65536; h++) {
        c.one(h << 16);                                                          // bf16
        const uint32_t sign = (h & 0x8000u) << 16, e = (h >> 10) & 31u, m = h & 1023u;
        uint32_t bits;
        if (e == 31) bits = sign | 0x7f800000u | (m << 13);
        else if (e) bits = sign | ((e + 112u) << 23) | (m << 13);
        else if (m) { float f = (float)m * 5.9604644775390625e-08f; bits = f2u(f) | sign; }
        else bits = sign;
        c.one(bits);                                                             // f16
    }
    // breakpoints of the algorithms, with their neighbours
    const uint32_t marks[] = {0x00000000u, 0x24000000u, 0x33000000u, 0x3eb17218u, 0x3f800000u, 0x3F851592u, 0x4195b844u, 0x41b00000u,
                              0x42b00000u, 0x42b17218u, 0x42cff1b5u, 0x7f800000u, 0x7fc00000u, 0x00800000u, 0x007fffffu, 0x3f000000u};
    for (uint32_t mk : marks)
        for (int d = -64; d <= 64; d++) {
            c.one(mk + (uint32_t)d);
            c.one((mk + (uint32_t)d) ^ 0x80000000u);
        }
    printf("tanhf %llu expm1f %llu expf %llu logf %llu sinf %llu cosf %llu f2bf %llu checked %llu\n", c.tanh_bad, c.expm1_bad, c.exp_bad, c.log_bad, c.sin_bad,
           c.cos_bad, c.bf_bad, c.checked);
    return (c.tanh_bad | c.expm1_bad | c.exp_bad | c.log_bad | c.sin_bad | c.cos_bad | c.bf_bad) ? 1 : 0;
}
