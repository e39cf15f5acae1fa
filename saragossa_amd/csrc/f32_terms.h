// f32 factors as three bf16 terms (kernels_f32_prefill.hip); also compiles for the host.
#pragma once

#include <stdint.h>

namespace skv {

#ifdef __HIPCC__
#define SKV_BOTH __host__ __device__ __forceinline__
#else
#define SKV_BOTH inline
#endif

SKV_BOTH uint32_t f32_word(float x) { return __builtin_bit_cast(uint32_t, x); }
SKV_BOTH float word_f32(uint32_t w) { return __builtin_bit_cast(float, w); }

// upper halves of two words, the first in the low half
SKV_BOTH uint32_t upper_halves(uint32_t x, uint32_t y) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_perm(y, x, 0x07060302u);
#else
    return (x >> 16) | (y & 0xffff0000u);
#endif
}
// two values rounded to bf16 (nearest even), the first in the low half
SKV_BOTH uint32_t bf16_pair(float x, float y) {
#ifdef __HIP_DEVICE_COMPILE__
    typedef __attribute__((ext_vector_type(2))) float f2;
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{x, y}, b2));
#else
    auto round = [](float v) {
        const uint32_t b = f32_word(v);
        return v != v ? b | 0x400000u : b + 0x7fffu + ((b >> 16) & 1u);
    };
    return upper_halves(round(x), round(y));
#endif
}

// Two f32 values as three bf16 terms each, x = t0 + t1 + t2 exactly: the value rounded to nearest, what
// that leaves (16 bits and a sign) rounded to nearest, the rest (8 bits and a sign), so t1 is at most 2^-8 of x and t2
// 2^-17. (With t0 cut off instead, t1 reaches 2^-7 and t2 2^-16, and what the products below leave out 2^-22
// of a product.) A term can be inexact only where it is below the smallest bf16, 2^-133. Infinities, and values that
// round to one (above 3.39e38), have terms that are not numbers: whatever they are multiplied with becomes one.
SKV_BOTH void three_terms(float x, float y, uint32_t &t0, uint32_t &t1, uint32_t &t2) {
    t0 = bf16_pair(x, y);
    const float x1 = x - word_f32(t0 << 16), y1 = y - word_f32(t0 & 0xffff0000u);
    t1 = bf16_pair(x1, y1);
    t2 = upper_halves(f32_word(x1 - word_f32(t1 << 16)), f32_word(y1 - word_f32(t1 & 0xffff0000u)));
}

// The products of two factors of three terms that are kept, (left term, right term). The three left out are together at most
// 2^-24 of the product (2^-27.4 in the mean square over normal factors), like the rounding of one f32 product, and of
// either sign.
struct TermPair {
    int l, r;
};
constexpr TermPair TERMS[6] = {{0, 0}, {0, 1}, {1, 0}, {1, 1}, {2, 0}, {0, 2}};

} // namespace skv
