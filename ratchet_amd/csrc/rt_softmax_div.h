// The 16-bit softmax's short divisions e / s by a row sum, in portable C++ so that the same text can be compiled for the
// host and compared with the rounded division over all pairs (tests/softmax_division_check.cpp does).  The includer defines RT_FN,
// the function qualifiers.  rinv is 1.0f / s; e is the exp value of one of the sum's terms.  The streaming kernel takes the short form for sums
// in [MIN, MAX] and divides by the others; the one with several rows to a wave takes it for every sum > 0: those below MIN as they are in
// f16, and in bf16 those outside after multiplying both sides by `scale`.
#ifndef RT_SOFTMAX_DIV_H
#define RT_SOFTMAX_DIV_H

// f16: e * rinv + e * rlow, where rinv + rlow is 1 / s to 48 bits, so the f32 quotient is off by one rounding.  Two 11-bit
// significands never divide to the middle between two f16 values and stay 2^-23 away from it, so f16 of that quotient is f16 of
// e / s (subnormal results too: their middles are exact f32 values; subnormal sums too, which are normal in f32, as 1 / s is).
struct ShortDivF16 {
    static constexpr float MIN = 6.103515625e-05f, MAX = 65504.0f;
    static constexpr bool TWO = true;                        // rlow is used
    static RT_FN float low(float s, float rinv) { return __builtin_fmaf(-s, rinv, 1.0f) * rinv; }
    static RT_FN float quotient(float e, float rinv, float rlow) { return __builtin_fmaf(e, rinv, __builtin_fmaf(e, rlow, 0.0f)); }
};

// bf16: e * (1 / s) is within 2^-23 of the quotient, and the quotient of two 8-bit significands is no closer than 2^-17 to the
// middle between two bf16 values (and never on it), or, where the result is subnormal, an exact f32 value when it is on the middle.
// Both sides times scale(s): s lies in [MIN, MAX] then, and a value that is no longer exact has a quotient of 0 with or without it.
struct ShortDivBf16 {
    static constexpr float MIN = 0x1p-100f, MAX = 0x1p100f;
    static constexpr bool TWO = false;
    static RT_FN float scale(float s) { return s < MIN ? 0x1p64f : s > MAX ? 0x1p-64f : 1.0f; }
    static RT_FN float low(float, float) { return 0.0f; }
    static RT_FN float quotient(float e, float rinv, float) { return e * rinv; }
};

#endif
