// FP8 E4M3FN unit-scale codec on the device (gfx950).
//
// Decode replaces fp8_e4m3x8_to_bf16x8 of the reference's shaders (crates/inference-backend-metal/src/components/
// metal/gqa_fp8.metal:1-25); encode replaces bf16_to_fp8_e4m3 of the page writer (.../metal/gqa_kv_page_write.metal:5-31,
// components/gqa/fp8.rs:19-45): round to nearest even, finite and infinite inputs saturate to +/-448 (0x7e), NaN keeps
// the E4M3FN NaN code (0x7f).  Every E4M3FN value is exactly representable in bf16, so decoding is exact.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_math.hip.h"

namespace khm {

// Two E4M3FN codes (the low or the high half of `codes`) to two bf16 values in one 32-bit word.  gfx950 converts OCP
// FP8 in hardware; the scale operand is a power of two and 1.0 leaves the value unchanged.
template <bool HIGH_HALF>
__device__ __forceinline__ uint32_t fp8x2_to_bf16x2(uint32_t codes) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(codes, 1.0f, HIGH_HALF));
}

// Eight codes (two words) to eight bf16 (four words), element order preserved.
__device__ __forceinline__ uint4 fp8x8_to_bf16x8(uint2 codes) {
    return make_uint4(fp8x2_to_bf16x2<false>(codes.x), fp8x2_to_bf16x2<true>(codes.x), fp8x2_to_bf16x2<false>(codes.y),
                      fp8x2_to_bf16x2<true>(codes.y));
}

// ---- FP8 matrix products with a split operand --------------------------------------------------------------------------
// v_mfma_scale_f32_16x16x128_f8f6f4 takes the page codes as they are, at twice the rate of the bf16 form.  The other operand is a
// sum of E4M3 pieces, each 2^-4 of the one before: piece n holds value * 2^(4 n), and its product carries the block scale 2^(-4 n).
typedef int i32x8 __attribute__((ext_vector_type(8)));
constexpr float kPieceStep = 0x1p-4f;
constexpr int kPieceScale0 = 0x7f7f7f7f, kPieceScale1 = 0x7b7b7b7b, kPieceScale2 = 0x77777777;   // E8M0: 2^0, 2^-4, 2^-8

// a register whose contents do not matter: the conversions fill one half of theirs at a time, and a zero would be an instruction
__device__ __forceinline__ int any_bits() {
    int bits;
    asm volatile("" : "=v"(bits));   // volatile: one for each use, not one register copied about
    return bits;
}
__device__ __forceinline__ uint32_t f32x4_to_fp8x4(float a, float b, float c, float d) {
    const int low = __builtin_amdgcn_cvt_pk_fp8_f32(a, b, any_bits(), false);
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, d, low, true);
}
// codes of x / scale (scale a power of two)
__device__ __forceinline__ uint32_t f32x4_to_scaled_fp8x4(float a, float b, float c, float d, float scale) {
    typedef short S16x2 __attribute__((ext_vector_type(2)));
    const S16x2 low = __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(__builtin_bit_cast(S16x2, any_bits()), a, b, scale, false);
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(low, c, d, scale, true));
}
// what the codes leave of x (exact: the remainder of a rounding)
__device__ __forceinline__ void subtract_fp8x4(float (&x)[4], uint32_t codes) {
    const auto low = __builtin_amdgcn_cvt_pk_f32_fp8((int)codes, false), high = __builtin_amdgcn_cvt_pk_f32_fp8((int)codes, true);
    x[0] -= low[0];
    x[1] -= low[1];
    x[2] -= high[0];
    x[3] -= high[1];
}
__device__ __forceinline__ void subtract_scaled_fp8x4(float (&x)[4], uint32_t codes, float scale) {
    const auto low = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(codes, scale, false), high = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(codes, scale, true);
    x[0] -= low[0];
    x[1] -= low[1];
    x[2] -= high[0];
    x[3] -= high[1];
}
// c + A . (B * scale): A are page codes, B one piece
__device__ __forceinline__ f32x4 mfma_fp8_k128(i32x8 a, i32x8 b, f32x4 c, int piece_scale) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, kPieceScale0, 0, piece_scale);
}

// A row of bf16 values as two pieces: scaled by a power of two so that the row's largest value lies in [2^7, 2^8), a value is four
// significant bits and a remainder of at most eight of its own units, both exact from 2^-14 of the largest on.  A row with an
// infinity keeps the signs of the infinite values, beside which the finite ones are nothing, and has an infinite scale; a NaN
// stays one.
struct SplitScale {
    float unit;      // the power of two a code is worth
    bool infinite;
    __device__ __forceinline__ float column_scale() const { return infinite ? INFINITY : unit; }
};
struct SplitCodes {
    uint2 high, low;
};
// the two bf16 magnitudes of `largest` and eight more, the larger of each position
__device__ __forceinline__ uint32_t largest_magnitudes(uint4 bits, uint32_t largest) {
    typedef unsigned short U16x2 __attribute__((ext_vector_type(2)));
    const uint32_t words[4] = {bits.x, bits.y, bits.z, bits.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
        largest = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(U16x2, words[i] & 0x7fff7fffu), __builtin_bit_cast(U16x2, largest)));
    return largest;
}
__device__ __forceinline__ uint32_t larger_half(uint32_t pair) { return (pair & 0xffffu) > (pair >> 16) ? (pair & 0xffffu) : (pair >> 16); }
__device__ __forceinline__ SplitScale split_scale_of(uint32_t largest_magnitude) {
    uint32_t exponent = largest_magnitude >> 7;
    exponent = exponent < 16u ? 16u : (exponent > 254u ? 254u : exponent);   // the unit and a sixteenth of it are normal numbers
    return SplitScale{__uint_as_float((exponent - 7u) << 23), largest_magnitude == 0x7f80u};
}
__device__ __forceinline__ SplitCodes split_bf16x8(uint4 bits, const SplitScale& scale) {
    typedef short S16x2 __attribute__((ext_vector_type(2)));
    uint32_t words[4] = {bits.x, bits.y, bits.z, bits.w};
    if (__builtin_amdgcn_ballot_w64(scale.infinite) != 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (!scale.infinite) continue;
            // 2^127 = 128 units of such a row (its exponent counts as 254)
            const uint32_t low = (words[i] & 0x7fffu) == 0x7f80u ? (words[i] & 0x8000u) | 0x7f00u : 0u;
            const uint32_t high = ((words[i] >> 16) & 0x7fffu) == 0x7f80u ? ((words[i] >> 16) & 0x8000u) | 0x7f00u : 0u;
            words[i] = low | (high << 16);
        }
    }
    uint32_t high[2], low[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const S16x2 first = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(__builtin_bit_cast(S16x2, any_bits()), __builtin_bit_cast(bf16x2, words[2 * i]), scale.unit, false);
        high[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(first, __builtin_bit_cast(bf16x2, words[2 * i + 1]), scale.unit, true));
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = j & 1 ? __uint_as_float(words[2 * i + j / 2] & 0xffff0000u) : bf16_bits_to_f32(words[2 * i + j / 2]);
        subtract_scaled_fp8x4(x, high[i], scale.unit);
        low[i] = f32x4_to_scaled_fp8x4(x[0], x[1], x[2], x[3], scale.unit * kPieceStep);
    }
    return SplitCodes{make_uint2(high[0], high[1]), make_uint2(low[0], low[1])};
}

// One bf16 bit pattern to its E4M3FN code, in integer arithmetic on the bf16 fields (7-bit mantissa -> 3 bits).
__device__ __forceinline__ uint32_t bf16_bits_to_fp8_e4m3fn(uint32_t bits) {
    const uint32_t sign = (bits >> 8) & 0x80u;
    const uint32_t magnitude = bits & 0x7fffu;
    if (magnitude > 0x7f80u) return sign | 0x7fu;             // NaN
    if (magnitude >= 0x43e0u) return sign | 0x7eu;            // >= 448 or infinite: saturate
    const uint32_t exponent = magnitude >> 7;                 // biased by 127
    if (exponent < 121u) {                                    // below 2^-6: E4M3FN subnormal, step 2^-9
        const float scaled = __uint_as_float(magnitude << 16) * 512.0f;
        const uint32_t mantissa = (uint32_t)__builtin_rintf(scaled);   // round half to even
        return sign | (mantissa < 8u ? mantissa : 8u);
    }
    uint32_t kept = (magnitude >> 4) & 0x7u;
    const uint32_t dropped = magnitude & 0xfu;
    uint32_t encoded_exponent = exponent - 120u;              // (exponent - 127) + 7
    if (dropped > 8u || (dropped == 8u && (kept & 1u))) ++kept;
    if (kept == 8u) {
        kept = 0u;
        ++encoded_exponent;
    }
    if (encoded_exponent > 15u || (encoded_exponent == 15u && kept >= 7u)) return sign | 0x7eu;
    return sign | (encoded_exponent << 3) | kept;
}

// Two bf16 bit patterns (low and high half of `pair`) to their two E4M3FN codes, written to the low (HIGH_HALF = false)
// or high 16 bits of `old` through v_cvt_scalef32_pk_fp8_bf16 with scale 1 (round to nearest even, subnormals below
// 2^-6).  The converter does not saturate (magnitudes above 464 come out as the NaN code), so magnitudes are clamped to
// 448 first, as 16-bit integers on the bf16 fields, which orders finite and infinite magnitudes alike; NaN would be
// clamped with them and is patched afterwards: it keeps its sign and becomes 0x7f.  Checked against the integer encoder
// above and the host codec over all 65 536 patterns in every position.
typedef unsigned short Fp8U16x2 __attribute__((ext_vector_type(2)));
typedef short Fp8I16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 Fp8Bf16x2 __attribute__((ext_vector_type(2)));

template <bool HIGH_HALF>
__device__ __forceinline__ uint32_t bf16x2_bits_to_fp8x2_no_nan(uint32_t old, uint32_t pair) {
    const Fp8U16x2 magnitude = __builtin_bit_cast(Fp8U16x2, pair & 0x7fff7fffu);
    const Fp8U16x2 limit = {0x43e0, 0x43e0};
    const uint32_t clamped = (pair & 0x80008000u) | __builtin_bit_cast(uint32_t, __builtin_elementwise_min(magnitude, limit));
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(__builtin_bit_cast(Fp8I16x2, old),
                                                                                 __builtin_bit_cast(Fp8Bf16x2, clamped), 1.0f, HIGH_HALF));
}

// Nonzero in the half of the result whose half of `pair` is a NaN.
__device__ __forceinline__ uint32_t bf16x2_nan_halves(uint32_t pair) {
    const Fp8U16x2 magnitude = __builtin_bit_cast(Fp8U16x2, pair & 0x7fff7fffu);
    const Fp8U16x2 infinity = {0x7f80, 0x7f80};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(magnitude, infinity));
}

__device__ __forceinline__ uint32_t bf16x2_bits_to_fp8x2_e4m3fn(uint32_t pair) {
    uint32_t codes = bf16x2_bits_to_fp8x2_no_nan<false>(0u, pair) & 0xffffu;
    const uint32_t nan = bf16x2_nan_halves(pair);
    if (nan != 0u) {
        if ((nan & 0xffffu) != 0u) codes = (codes & 0xff00u) | ((pair >> 8) & 0x80u) | 0x7fu;
        if ((nan >> 16) != 0u) codes = (codes & 0x00ffu) | ((pair >> 16) & 0x8000u) | 0x7f00u;
    }
    return codes;
}

// Four bf16 bit patterns (`first` holds elements 0 and 1, `second` elements 2 and 3) to four codes in element order.
__device__ __forceinline__ uint32_t bf16x4_bits_to_fp8x4_e4m3fn(uint32_t first, uint32_t second) {
    uint32_t codes = bf16x2_bits_to_fp8x2_no_nan<true>(bf16x2_bits_to_fp8x2_no_nan<false>(0u, first), second);
    const uint32_t nan_first = bf16x2_nan_halves(first), nan_second = bf16x2_nan_halves(second);
    if ((nan_first | nan_second) != 0u) {
        if ((nan_first & 0xffffu) != 0u) codes = (codes & 0xffffff00u) | ((first >> 8) & 0x80u) | 0x7fu;
        if ((nan_first >> 16) != 0u) codes = (codes & 0xffff00ffu) | ((first >> 16) & 0x8000u) | 0x7f00u;
        if ((nan_second & 0xffffu) != 0u) codes = (codes & 0xff00ffffu) | ((second << 8) & 0x800000u) | 0x7f0000u;
        if ((nan_second >> 16) != 0u) codes = (codes & 0x00ffffffu) | (second & 0x80000000u) | 0x7f000000u;
    }
    return codes;
}

// Eight bf16 bit patterns to eight codes, element order preserved.
__device__ __forceinline__ uint2 bf16x8_bits_to_fp8x8_e4m3fn(uint4 bits) {
    return make_uint2(bf16x4_bits_to_fp8x4_e4m3fn(bits.x, bits.y), bf16x4_bits_to_fp8x4_e4m3fn(bits.z, bits.w));
}

}  // namespace khm
