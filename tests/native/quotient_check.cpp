// CPU check of corrected_quotient (economize_amd/csrc/fp8_codec.hpp) against IEEE division where the kernels use it.
// Prints the number of differences, which must be 0.
#include <cstdio>
#include <initializer_list>

#include "../../economize_amd/csrc/fp8_codec.hpp"

namespace {

// n / levels over every significand (an exponent more or less changes no bit of the comparison).
long constant_divisors() {
    long bad = 0;
    for (const float levels : {3.0f, 15.0f})
        for (uint32_t m = 0; m < 1u << 23; ++m) {
            const float n = eco::bits_f32(0x3F800000u | m);
            bad += eco::corrected_quotient(n, levels, 1.0f / levels) != n / levels;
        }
    return bad;
}

// round_half_even(n / s) for every 11-bit s and n within two ulps of h * s, h every half integer up to 14.5, with a
// reciprocal off by up to an ulp either way.
long codes() {
    long bad = 0;
    for (uint32_t ms = 0; ms < 1u << 10; ++ms) {
        const float s = eco::bits_f32(0x3F800000u | ms << 13);
        for (int twice = 1; twice < 30; twice += 1)
            for (int off = -2; off <= 2; ++off)
                for (int r_off = -1; r_off <= 1; ++r_off) {
                    const float n = eco::bits_f32(eco::f32_bits(0.5f * twice * s) + off);
                    const float r = eco::bits_f32(eco::f32_bits(1.0f / s) + r_off);
                    bad += rintf(eco::corrected_quotient(n, s, r)) != rintf(n / s);
                }
    }
    return bad;
}

// x / s for every 11-bit x (the 8-bit ones among them) and every s, with the rounded reciprocal: blocks of s that stay in
// the cache, vectorised over s.
long shared_scales() {
    constexpr int kBlock = 2048;
    long bad = 0;
#pragma omp parallel for reduction(+ : bad)
    for (uint32_t block = 0; block < (1u << 23) / kBlock; ++block) {
        float s[kBlock], r[kBlock];
        for (int i = 0; i < kBlock; ++i) {
            s[i] = eco::bits_f32(0x3F800000u | (block * kBlock + i));
            r[i] = 1.0f / s[i];
        }
        for (uint32_t mx = 0; mx < 1u << 10; ++mx) {
            const float x = eco::bits_f32(0x3F800000u | mx << 13);
            int differ = 0;
            for (int i = 0; i < kBlock; ++i) differ += eco::corrected_quotient(x, s[i], r[i]) != x / s[i];
            bad += differ;
        }
    }
    return bad;
}

}  // namespace

int main() {
    std::printf("%ld\n", constant_divisors() + codes() + shared_scales());
    return 0;
}
