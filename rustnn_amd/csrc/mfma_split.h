// fp32 products on the bf16 matrix cores.
//
// A float with 24 significant bits is the exact sum of three bf16 values of 8
// bits each: its leading 8 bits, those of the remainder, and the rest (cut
// off, not rounded, so that the largest float's leading part stays finite).
// Of the nine part products of a x b the three smallest (mid lo, lo mid, lo
// lo) are left out; the other six are exact in the matrix core and summed in
// its fp32 accumulator, sixteen k values and two roundings an instruction where
// v_mfma_f32_32x32x2f32 takes two.  What is left out is below 2^-21 of the
// product with both operands cut off (mid < 2^-7, lo < 2^-15 of the leading
// bit), always of the product's sign, so that it adds up over k; below 2^-22
// and of no common sign with one operand's leading part rounded to nearest
// instead (|mid| <= 2^-8, |lo| < 2^-16), as every caller does.
//
// Measured on MI355X.  Rate: the bf16 pipe sustains 1.79 PFLOP/s from
// registers, six products 298 TFLOP/s of fp32 work against the fp32 pipe's
// 154; with the splitting of both operands in the same wave 200-220.  Error
// against f64 over random normal operands (fp32 pipe / split): K = 16 8.0e-8
// / 7.0e-8, K = 256 3.1e-7 / 2.4e-7, K = 4096 1.20e-6 / 1.11e-6.  The sum inside one instruction is cut off
// toward -inf, which leaves a mean error of -1.4e-8 (K = 256) to -5e-8 (K =
// 1024) of the result's size where the fp32 pipe has none above 3e-9: it adds
// up where many results are summed (a bias gradient over 8192 rows was 4
// times further off).  Two ways out, both with a mean error below 2e-9: a
// second accumulator for the five smaller products (K = 256 1.1e-7, K = 1024
// 1.9e-7 against the fp32 pipe's 5.6e-7), or, where registers are short, half
// of the k steps accumulating the negated product (K = 256 1.8e-7).
//
// The parts of a value below 2^-110 would be denormal bf16, which end at
// 2^-133 (1e-36 kept 13 bits, 1e-41 none), so a split multiplies by BF3_UP
// first: the last bit of the smallest denormal float becomes 2^-125.  Sums of
// products are multiplied by BF3_DOWN when they are complete.  Operands from
// 2^104 and sums from 2^80 (1.2e24) on overflow this way and are taken again
// by the callers as every result that is not finite.  The multiplies cost
// 8192 x 256 x 768 28.2 -> 28.6 us, 4096^3 779 -> 785, 3x3 32 -> 32 @32x32 at
// batch 128 23.0 -> 23.2 and its dW 25.0 -> 26.2.
#pragma once

#include "rnn_internal.h"

#include <type_traits>

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float BF3_UP = 0x1p24f, BF3_DOWN = 0x1p-48f;

// The parts of 8 floats times BF3_UP, as operands of v_mfma_f32_32x32x16_bf16.
struct Bf3 {
    u32x4 hi, mid, lo;
};

// Two floats' leading 16 bits in one register.
__device__ __forceinline__ uint32_t bf3_top2(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float bf3_rest(float a) {
    return a - __uint_as_float(__float_as_uint(a) & 0xFFFF0000u);
}

// up: BF3_UP or -BF3_UP (the negated product).
__device__ __forceinline__ Bf3 bf3_split(const float (&x)[8], float up = BF3_UP) {
    Bf3 p;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float a = x[2 * j] * up, b = x[2 * j + 1] * up;
        p.hi[j] = bf3_top2(a, b);
        const float ra = bf3_rest(a), rb = bf3_rest(b);
        p.mid[j] = bf3_top2(ra, rb);
        p.lo[j] = bf3_top2(bf3_rest(ra), bf3_rest(rb));
    }
    return p;
}

// The parts rounded to nearest instead of cut off: with one operand of a
// product split this way the part products left out have no common sign (cut
// off, they make results 3.3e-8 smaller).  Slower (bf16 conversions), and
// values within 2^-9 of the largest float overflow to infinity.
__device__ __forceinline__ Bf3 bf3_split_round(const float (&x)[8]) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    Bf3 p;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float a = x[2 * j] * BF3_UP, b = x[2 * j + 1] * BF3_UP;
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const bf16x2 v = {(__bf16)a, (__bf16)b};
            const uint32_t u = __builtin_bit_cast(uint32_t, v);
            (q == 0 ? p.hi : q == 1 ? p.mid : p.lo)[j] = u;
            a -= __uint_as_float(u << 16);
            b -= __uint_as_float(u & 0xFFFF0000u);
        }
    }
    return p;
}

// The same with the leading part alone rounded, which already takes the common
// sign away (1 + 2^-7 - 2^-23 squared: 4.7e-7 too small cut off, 2e-9 this way;
// sums of positive products at any k 4.1e-8 / below 1e-9).  On the weights
// of the 3x3 convolutions: logits of 17 ResNets of 8 to 20 layers 1.047 times
// the fp32 pipe's error against 64 bits cut off, 0.996 this way, for 1% of the
// time (a ResNet-20 step 1953 -> 1973 us).  CVT: rounded by a bf16 conversion
// (ties to even) instead of an integer add (away from zero), three
// instructions a pair of floats less and a longer chain: 512^3 (32 x 64 tiles)
// 9.5 us against 10.1, 2048^3 (128 x 128) 118.6 against 116.2.
// An infinity's or NaN's remainder is a NaN.
template <bool CVT = false>
__device__ __forceinline__ Bf3 bf3_split_near(const float (&x)[8], float up = BF3_UP) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    Bf3 p;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float xa = x[2 * j] * up, xb = x[2 * j + 1] * up;
        float a, b;  // the leading parts
        if constexpr (CVT) {
            const bf16x2 v = {(__bf16)xa, (__bf16)xb};
            const uint32_t u = __builtin_bit_cast(uint32_t, v);
            p.hi[j] = u;
            a = __uint_as_float(u << 16);
            b = __uint_as_float(u & 0xFFFF0000u);
        } else {
            a = __uint_as_float((__float_as_uint(xa) + 0x8000u) & 0xFFFF0000u);
            b = __uint_as_float((__float_as_uint(xb) + 0x8000u) & 0xFFFF0000u);
            p.hi[j] = bf3_top2(a, b);
        }
        const float ra = xa - a, rb = xb - b;
        p.mid[j] = bf3_top2(ra, rb);
        p.lo[j] = bf3_top2(bf3_rest(ra), bf3_rest(rb));
    }
    return p;
}

__device__ __forceinline__ f32x16 bf3_mfma1(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x4 bf3_mfma1(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Calls f(pick, small) for each of the six part products, smallest first;
// pick(a, b, c) adds that product of two fragments to accumulator c; small is
// 0 for the product of the leading parts, 1 for the others.
template <typename F>
__device__ __forceinline__ void bf3_products(F &&f) {
    const std::integral_constant<int, 0> lead;
    const std::integral_constant<int, 1> small;
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.mid, b.mid, c); }, small);
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.hi, b.lo, c); }, small);
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.lo, b.hi, c); }, small);
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.hi, b.mid, c); }, small);
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.mid, b.hi, c); }, small);
    f([](const Bf3 &a, const Bf3 &b, auto c) { return bf3_mfma1(a.hi, b.hi, c); }, lead);
}

template <int TM, int TN>
__device__ __forceinline__ void bf3_negate(f32x16 (&acc)[TM][TN]) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) acc[i][j] = -acc[i][j];
}

// Whether a value is an infinity or a NaN.
__device__ __forceinline__ bool bf3_nonfinite(float c) {
    return __builtin_amdgcn_classf(c, 0x207);
}
