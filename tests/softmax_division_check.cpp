// Host check of the 16-bit softmax's short divisions (ratchet_amd/csrc/rt_softmax_div.h, the kernels' own text): for every exp
// value e >= 0 and every `stride`-th row sum s inside the range where the streaming kernel takes them, and for every e <= s and every
// s > 0 outside of it, where the kernel with several rows to a wave takes them too, the short form must round to the
// bits of the correctly rounded f32 quotient rounded to the 16-bit type, which is what the reference's half types compute.
// Build: g++ -O2 -std=c++17 -ffp-contract=off -mfma -I ratchet_amd/csrc.   Usage: softmax_division_check STRIDE
// prints "f16 <n> bf16 <n> checked <m>" (n: pairs that differ), exit code 0 iff both are 0.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#define RT_FN inline
#include "rt_softmax_div.h"

static float u2f(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static uint32_t f2u(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static uint16_t to_bf16(float f) {                            // finite, nearest even
    const uint32_t u = f2u(f);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}
static float from_f16(uint16_t h) {                           // h >= 0, finite
    return (h & 0x7c00) ? u2f(((uint32_t)h << 13) + 0x38000000u) : (float)h * 0x1p-24f;
}
static uint16_t to_f16(float f) {                             // 0 <= f, nearest even
    if (f >= 65520.0f) return 0x7c00;
    if (f < 0x1p-14f) return (uint16_t)(f2u(f + 0.5f) - 0x3f000000u);      // one f32 step of [0.5, 1) is 2^-24, a subnormal f16 step
    const uint32_t u = f2u(f);
    return (uint16_t)((u + 0xfffu + ((u >> 13) & 1u) - 0x38000000u) >> 13);
}

int main(int argc, char** argv) {
    const unsigned stride = argc > 1 ? (unsigned)strtoul(argv[1], nullptr, 10) : 1;
    unsigned long long bad16 = 0, badbf = 0, checked = 0;
    for (uint32_t sb = 1; sb < 0x7c00; sb += stride) {
        const float s = from_f16((uint16_t)sb), rinv = 1.0f / s, rlow = ShortDivF16::low(s, rinv);
        const uint32_t last = s < ShortDivF16::MIN ? sb : 0x7bff;             // (a sum is never below its terms)
        for (uint32_t eb = 0; eb <= last; eb++) {
            const float e = from_f16((uint16_t)eb);
            bad16 += to_f16(ShortDivF16::quotient(e, rinv, rlow)) != to_f16(e / s);
            checked++;
        }
    }
    for (uint32_t sb = 1; sb < 0x7f80; sb += stride) {
        const float sum = u2f(sb << 16), by = ShortDivBf16::scale(sum), s = sum * by, rinv = 1.0f / s, rlow = ShortDivBf16::low(s, rinv);
        if (s < ShortDivBf16::MIN || s > ShortDivBf16::MAX) return 2;
        if (by != 1.0f) {
            for (uint32_t eb = 0; eb <= sb; eb++) {
                const float e = u2f(eb << 16);
                badbf += to_bf16(ShortDivBf16::quotient(u2f((uint32_t)to_bf16(e * by) << 16), rinv, rlow)) != to_bf16(e / sum);
                checked++;
            }
            continue;
        }
        for (uint32_t eb = 0; eb < 0x7f80; eb++) {
            const float e = u2f(eb << 16), q = e / s;
            if (std::isinf(q)) break;                         // a sum is never below its terms
            badbf += to_bf16(ShortDivBf16::quotient(e, rinv, rlow)) != to_bf16(q);
            checked++;
        }
    }
    printf("f16 %llu bf16 %llu checked %llu\n", bad16, badbf, checked);
    return bad16 || badbf;
}
