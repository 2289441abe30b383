// vedic_split.hpp -- binary32 values as exact sums of three bf16 values.
//
// gfx950's matrix cores multiply bf16 sixteen times as fast as binary32, and a
// binary32 significand (24 bits) is exactly three bf16 significands (8 bits
// each): x = x1 + x2 + x3 with x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 - x2
// (round to nearest even, every difference exact; |x2| <= 2^-8 |x|, |x3| <=
// 2^-17 |x|).  A product then is
//     x y = x1 y1 + (x1 y2 + x2 y1) + (x1 y3 + x3 y1 + x2 y2) + r,
// six bf16 products, each exact in the MFMA's binary32 accumulation, and
// |r| <= |x2 y3| + |x3 y2| + |x3 y3| <= 2^-24 (1 + 2^-10) |x y|: as much as one
// binary32 rounding at worst (x = y = 1 + 2^-8 - 2^-17 loses 0.99 of it), made
// good by rounding sums once per 16 steps (Henry, Tang, Heinecke, "Leveraging
// the bfloat16 artificial intelligence datatype for higher-precision
// computations", ARITH 2019).  Six bf16 MFMAs cover 16 contraction steps in the
// time v_mfma_f32_32x32x2_f32 covers 6: 2.67 times the binary32 rate.
//
// Measured against float64 (32 x 32 tiles, K contraction steps, relative
// 2-norm, six-product sums / v_mfma_f32_32x32x2_f32): N(0,1) operands K = 16
// 3.4e-8 / 7.2e-8, 64 1.1e-7 / 1.4e-7, 1024 4.9e-7 / 5.7e-7, 8192 1.4e-6 /
// 1.6e-6; uniform [0,1) 3.2e-8 / 6.2e-8, 8.4e-8 / 1.2e-7, 2.9e-7 / 4.3e-7,
// 7.5e-7 / 1.2e-6; softmax rows times N(0,1) as the first.
//
// Range.  The bf16 MFMA flushes subnormal operands, so values are scaled by
// 2^24 before the split: the last bit of any binary32 value, the smallest
// subnormal (2^-149) included, then is at least 2^-125 and every part is zero
// or normal.  (The attention kernels distribute the factors as their sums
// need them.)  A value that rounds to 2^104 or more in bf16, an infinity or a
// NaN makes the parts, and so the sums they enter, infinite or NaN; so does a
// scaled sum of 2^128 or more.  The kernels check their sums for that and repeat
// such a block with v_mfma_f32_32x32x2_f32 on the unscaled values.
#pragma once

#include "vedic_common.hpp"

namespace vedic {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));

constexpr float kSplitScale = 16777216.0f;                         // 2^24, on each operand
constexpr float kSplitUnscale = 1.0f / 16777216.0f;                // 2^-24
constexpr float kSplitUnscale2 = kSplitUnscale * kSplitUnscale;    // 2^-48, on a product of two scaled operands

// The three parts of a pair of (scaled) values, packed.
struct SplitPair {
    uint32_t p[3];
};

// (v_dot2_f32_bf16 with (-1, 0) would take x - b in one instruction instead of
// an unpack and a subtraction, but it holds up the matrix pipe: four of them
// beside each 32-cycle MFMA made it 66 cycles, four v_fma_f32 none.)
__device__ __forceinline__ SplitPair split_pair(float x, float y) {
    SplitPair s;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const bf16x2_t b = __builtin_convertvector((float2_t{x, y}), bf16x2_t);
        s.p[i] = __builtin_bit_cast(uint32_t, b);
        if (i < 2) {
            x -= __builtin_bit_cast(float, s.p[i] << 16);
            y -= __builtin_bit_cast(float, s.p[i] & 0xFFFF0000u);
        }
    }
    return s;
}

// Three bf16x8 MFMA operands, part by part.
struct SplitFrag {
    bf16x8_t p[3];
};

// The same of scale x and scale y: the first remainder is taken from the exact
// product, spelled out so that every kernel splits a value alike (the compiler
// would contract the multiplication into the subtraction in some and not in
// others, and scores that two kernels compute for one probability would differ).
__device__ __forceinline__ SplitPair split_pair(float x, float y, float scale) {
    SplitPair s;
    s.p[0] = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t{x * scale, y * scale}), bf16x2_t));
    x = __builtin_fmaf(x, scale, -__builtin_bit_cast(float, s.p[0] << 16));
    y = __builtin_fmaf(y, scale, -__builtin_bit_cast(float, s.p[0] & 0xFFFF0000u));
    s.p[1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t{x, y}), bf16x2_t));
    x -= __builtin_bit_cast(float, s.p[1] << 16);
    y -= __builtin_bit_cast(float, s.p[1] & 0xFFFF0000u);
    s.p[2] = __builtin_bit_cast(uint32_t, __builtin_convertvector((float2_t{x, y}), bf16x2_t));
    return s;
}

// Eight values -> their parts.
__device__ __forceinline__ SplitFrag split8(const float (&v)[8]) {
    u32x4_t w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const SplitPair s = split_pair(v[2 * e], v[2 * e + 1]);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p][e] = s.p[p];
    }
    SplitFrag f;
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p] = __builtin_bit_cast(bf16x8_t, w[p]);
    return f;
}

__device__ __forceinline__ SplitFrag split8(const float (&v)[8], float scale) {
    u32x4_t w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const SplitPair s = split_pair(v[2 * e], v[2 * e + 1], scale);
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p][e] = s.p[p];
    }
    SplitFrag f;
#pragma unroll
    for (int p = 0; p < 3; ++p) f.p[p] = __builtin_bit_cast(bf16x8_t, w[p]);
    return f;
}

// The six products in ascending size: the small ones meet the accumulator
// first.
constexpr int kSplitProducts = 6;
__device__ constexpr int kSplitA[kSplitProducts] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kSplitB[kSplitProducts] = {0, 2, 1, 0, 1, 0};

// acc += a . b over 16 contraction steps.
__device__ __forceinline__ float16_t mfma_split(const SplitFrag& a, const SplitFrag& b, float16_t acc) {
#pragma unroll
    for (int q = 0; q < kSplitProducts; ++q)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[kSplitA[q]], b.p[kSplitB[q]], acc, 0, 0, 0);
    return acc;
}

// The same with the roles of a and b exchanged: b . a has these bits.
__device__ __forceinline__ float16_t mfma_split_swapped(const SplitFrag& a, const SplitFrag& b, float16_t acc) {
#pragma unroll
    for (int q = 0; q < kSplitProducts; ++q)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[kSplitB[q]], b.p[kSplitA[q]], acc, 0, 0, 0);
    return acc;
}

// NaN iff some accumulator is infinite or NaN.
__device__ __forceinline__ float nonfinite_probe(const float16_t& v, float t) {
#pragma unroll
    for (int e = 0; e < 16; ++e) t = __builtin_fmaf(v[e], 0.0f, t);
    return t;
}

}  // namespace vedic
