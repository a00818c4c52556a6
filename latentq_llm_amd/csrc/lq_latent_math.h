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

// Z -> residual nibble, and q = rint(Z) (half to even, as torch.round) plus the codec's carry as a saturated integer
// (NaN -> 0). The difference Z - q needs no rounding to bf16: Z has 8 significant bits, and its distance to the nearest
// integer is Z itself below a half and a multiple of Z's last place of at most a half above. An infinite Z leaves a NaN
// residual (nibble 0, no carry), and no Z above 2^23 carries, so the sum does not overflow.
__device__ __forceinline__ unsigned lq_latent_residual(float Z, const CodecParams &pq, unsigned &q_carry) {
    const float q = rintf(Z);
    bool carry;
    const unsigned nib = nibble_of_half(level_3fold(Z - q, pq), carry);
    unsigned qi;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(qi) : "v"(q));
    q_carry = qi + (carry ? 1u : 0u);
    return nib;
}

// One element of the re-quantiser: Z = bf16(bf16(t / s) + z), q = rint(Z), residual nibble and
// carry from bf16(Z - q), code = clamp(bf16(q + carry), 0, 15).
// Only bf16(t / s) is needed, and t and s are bf16 numbers: their quotient keeps a relative distance of at
// least 2^-17 from every bf16 rounding tie (a tie has a 9-bit odd significand, and s * tie = t has no solution
// with t below 2^8), so for 2^-40 <= s <= 2^40 (kFast; the caller branches once per group) the product
// t * RN(1/s), which is within 2^-23 of the quotient, rounds to the same bf16 number. Where the quotient is a
// bf16 subnormal that argument fails, and there q = rint(Z) and the residual level (0) are the same either way;
// infinities and NaN go the same way through the product as through the quotient.
template <bool kFast>
__device__ __forceinline__ void lq_latent_requant_elem(float t, float s, float z, float r, const CodecParams &pq,
                                                       unsigned &nib, unsigned &code) {
    const float quo = kFast ? t * r : t / s;
    const float Z = lq_bf16r(lq_bf16r(quo) + z);
    unsigned q;
    nib = lq_latent_residual(Z, pq, q);
    // clamp(bf16(q + carry), 0, 15): q + carry is an integer, bf16 keeps every integer up to 256 and is
    // monotonic, so the rounding cannot change what the clamp returns; a NaN ends as code 0
    code = lq_med3_i32<0, 15>(q);
}

// ---- 8-bit weights (int8 codes, one bf16 scale per row; utils/quant.py:88-103, 826-837, 1069-1070) ----
// latent = bf16(bf16(value(nibble)) * s) + bf16(q * s); the caller applies the last rounding
__device__ __forceinline__ float lq_latent_w8_value(unsigned byte, float value_bf16, float s) {
    const float q = (float)(int)(signed char)(byte & 0xFFu);
    return lq_bf16r(value_bf16 * s) + lq_bf16r(q * s);
}

// One element of the 8-bit re-quantiser: Z = bf16(t / s), q = rint(Z), residual nibble and carry from
// bf16(Z - q), code byte = clamp(q + carry, -128, 127) (NaN -> 0). kFast: the quotient as the product with
// r = 1 / s, valid for 2^-40 <= |s| <= 2^40 (see lq_latent_requant_elem).
template <bool kFast>
__device__ __forceinline__ void lq_latent_w8_requant_elem(float t, float s, float r, const CodecParams &pq, unsigned &nib,
                                                          unsigned &byte) {
    const float quo = kFast ? t * r : t / s;
    const float Z = lq_bf16r(quo);
    unsigned q;
    nib = lq_latent_residual(Z, pq, q);
    // q + carry is an integer (bf16 holds it exactly wherever the clamp does not decide); NaN -> 0
    byte = lq_med3_i32<-128, 127>(q) & 0xFFu;
}
