// Per-element arithmetic of the lbit = 4 latent weight (codes + 4-bit residual), shared by the
// latent passes (lq_latent.hip) and the fused optimizer step (lq_adam8.hip). Every line is one
// tensor operation of the reference's chains (utils/quant.py:45-72, 803-837) with its bf16 rounding.
#pragma once
#include "lq_common.h"
#include "lq_residual_codec.h"

// The dequantised value of a residual nibble depends on nothing but the nibble, so a workgroup keeps
// the 16 values bf16(value(n - 8)) in LDS and an element costs one LDS read instead of the curve's
// dozen selects and operations. Threads 0..15 fill the table; the caller synchronises before use.
__device__ __forceinline__ void lq_latent_fill_value_table(float *tab, const CodecParams &pd) {
    if (threadIdx.x < 16) tab[threadIdx.x] = lq_bf16r(value_3fold((int)threadIdx.x - 8, pd));
}

// Byte offsets into the table of the 8 nibbles of a residual word, element 0's the highest: lq_latent_value_of(tab, q, k) is element k's
// value. An element's offset is one byte of a word, where a shift and a mask for each took one more instruction.
struct lq_latent_offsets {
    unsigned even, odd;
};
__device__ __forceinline__ lq_latent_offsets lq_latent_value_offsets(unsigned residual) {
    return {(residual >> 2) & 0x3C3C3C3Cu, (residual << 2) & 0x3C3C3C3Cu};
}
__device__ __forceinline__ float lq_latent_value_of(const float *tab, const lq_latent_offsets &q, int k) {
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(tab) + (((k & 1 ? q.odd : q.even) >> (24 - 8 * (k >> 1))) & 0xFFu));
}

// The weight part bf16(bf16(q - z) * s) of the 8 elements of a code word: one fma each on the code read as an FP8 number
// where that equals the two roundings (integer z with |z| <= 240, s not extreme: q - z is exact in bf16, and the fma
// rounds the exact product once before the rounding to bf16 takes the rest), the two roundings otherwise.
__device__ __forceinline__ bool lq_latent_one_fma(float s, float z) {
    return (z == floorf(z)) && (fabsf(z) <= 240.0f) && (s >= 0x1p-100f) && (s <= 0x1p100f);
}
__device__ __forceinline__ void lq_latent_weights(unsigned word, float s, float z, bool one_fma, float (&w)[8]) {
    lq_dequant_word_f32(word, 512.0f * s, -(z * s), w);
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = lq_bf16r(w[k]);
    if (!one_fma) {
        asm volatile("; two roundings");  // (keeps this side from being computed along with the other one)
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = lq_bf16r(lq_bf16r((float)lq_code(word, k) - z) * s);
    }
}

// latent = bf16(bf16(bf16(value(nibble)) * s) + bf16(bf16(q - z) * s)) with value_bf16 =
// bf16(value(nibble)) from the table; the caller applies the last rounding
__device__ __forceinline__ float lq_latent_value(float weight, float value_bf16, float s) {
    return lq_bf16r(value_bf16 * s) + weight;
}

// min(max(v, LO), HI) of a signed integer
template <int LO, int HI>
__device__ __forceinline__ unsigned lq_med3_i32(unsigned v) {
    const int lo = (int)v < HI ? (int)v : HI;
    return (unsigned)(lo > LO ? lo : LO);
}

// byte SEL of `old` replaced by sat_u8(rne(v)) (a loop's index once it is unrolled)
__device__ __forceinline__ unsigned lq_put_u8(int sel, float v, unsigned old) {
    return sel == 0 ? act_cvt_pk_u8<0>(v, old) : sel == 1 ? act_cvt_pk_u8<1>(v, old) : sel == 2 ? act_cvt_pk_u8<2>(v, old) : act_cvt_pk_u8<3>(v, old);
}

// The residual of Z, q = rint(Z) (half to even, as torch.round): its nibble as a number (below 0 and NaN: nibble 0, by the saturating
// conversion that follows) and the codec's carry. The difference Z - q needs no rounding to bf16: Z has 8 significant bits, and its
// distance to the nearest integer is Z itself below a half and a multiple of Z's last place of at most a half above. An infinite Z
// leaves a NaN residual (nibble 0, no carry), and no Z above 2^23 carries. Without a carry the level is at most 7.
__device__ __forceinline__ float lq_latent_residual(float Z, float q, const CodecParams &pq, bool &carry) {
    const float lv = level_3fold<true>(Z - q, pq);
    carry = lv > 7.5f;
    return carry ? 1.0f : lv + 8.0f;
}

// The re-quantiser on 8 elements: Z = bf16(bf16(t / s) + z), q = rint(Z), residual nibble and carry from bf16(Z - q), code =
// clamp(bf16(q + carry), 0, 15) (NaN -> 0); to one code word and one residual word.
// Only bf16(t / s) is needed, and t and s are bf16 numbers: their quotient keeps a relative distance of at
// least 2^-17 from every bf16 rounding tie (a tie has a 9-bit odd significand, and s * tie = t has no solution
// with t below 2^8), so for 2^-40 <= s <= 2^40 (kFast; the caller branches once per group) the product
// t * RN(1/s), which is within 2^-23 of the quotient, rounds to the same bf16 number. Where the quotient is a
// bf16 subnormal that argument fails, and there q = rint(Z) and the residual level (0) are the same either way;
// infinities and NaN go the same way through the product as through the quotient.
// q + carry is an integer, bf16 keeps every integer up to 256 and is monotonic, so its rounding cannot change what the clamp returns.
// Nibbles go into bytes, elements 0, 2, .. and 1, 3, .. apart, by the conversion that saturates and inserts: 16 (q + carry) has the code
// in the upper half of its byte (240 and all that saturates: 15), and the two words are put together once for 8 elements. As
// integers they took two instructions more an element (curve parameters by value: by reference the compiler selects their addresses): optimizer step with int4 + residual, 50 M elements 133.8 -> 131.2 us.
template <bool kFast>
__device__ __forceinline__ void lq_latent_requant8(const float (&t)[8], float s, float z, float r, const CodecParams pq, unsigned &code_word,
                                                   unsigned &residual_word) {
    unsigned code[2] = {0u, 0u}, res[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float quo = kFast ? t[k] * r : t[k] / s;
        const float Z = lq_bf16r(lq_bf16r(quo) + z), q = rintf(Z);
        bool carry;
        const float nib = lq_latent_residual(Z, q, pq, carry);
        res[k & 1] = lq_put_u8(3 - (k >> 1), nib, res[k & 1]);
        code[k & 1] = lq_put_u8(k >> 1, fmaf(q, 16.0f, carry ? 16.0f : 0.0f), code[k & 1]);
    }
    code_word = (code[0] & 0xF0F0F0F0u) | ((code[1] >> 4) & 0x0F0F0F0Fu);
    residual_word = (res[0] << 4) | res[1];
}

// ---- 8-bit weights (int8 codes, one bf16 scale per row; utils/quant.py:88-103, 826-837, 1069-1070) ----
// latent = bf16(bf16(value(nibble)) * s) + bf16(q * s); the caller applies the last rounding
__device__ __forceinline__ float lq_latent_w8_value(unsigned byte, float value_bf16, float s) {
    const float q = (float)(int)(signed char)(byte & 0xFFu);
    return lq_bf16r(value_bf16 * s) + lq_bf16r(q * s);
}

// The 8-bit re-quantiser on 8 elements: Z = bf16(t / s), q = rint(Z), residual nibble and carry from bf16(Z - q), code byte =
// clamp(q + carry, -128, 127) (NaN -> 0, which a saturating conversion to unsigned bytes would not give). kFast: the quotient as
// the product with r = 1 / s, valid for 2^-40 <= |s| <= 2^40 (see lq_latent_requant8).
template <bool kFast>
__device__ __forceinline__ void lq_latent_w8_requant8(const float (&t)[8], float s, float r, const CodecParams pq, u32x2_t &codes,
                                                      unsigned &residual_word) {
    unsigned code[2] = {0u, 0u}, res[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float quo = kFast ? t[k] * r : t[k] / s;
        const float Z = lq_bf16r(quo), q = rintf(Z);
        bool carry;
        const float nib = lq_latent_residual(Z, q, pq, carry);
        res[k & 1] = lq_put_u8(3 - (k >> 1), nib, res[k & 1]);
        unsigned qi;  // q + carry is an integer (bf16 holds it exactly wherever the clamp does not decide)
        asm("v_cvt_i32_f32 %0, %1" : "=v"(qi) : "v"(q));
        code[k >> 2] |= (lq_med3_i32<-128, 127>(qi + (carry ? 1u : 0u)) & 0xFFu) << (8 * (k & 3));
    }
    codes = u32x2_t{code[0], code[1]};
    residual_word = (res[0] << 4) | res[1];
}
