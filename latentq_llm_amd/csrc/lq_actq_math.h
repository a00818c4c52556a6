// Arithmetic of the activation quantisers: shared by the passes of lq_actq.hip and the kernel that quantises a few tokens
// on its way into an int8 product (lq_gemv_i8.hip).
#pragma once
#include "lq_common.h"

// x8 = clamp(rne(bf16(bf16(x * 127) / clampv)), -128, 127); 8 elements per thread.
// The clamp value is the maximum of a bf16 tensor in every use the reference makes of it, i.e. a bf16 number;
// the quotient of two bf16 numbers keeps 2^-17 (relative) from every bf16 rounding tie, so bf16(a / c) is
// bf16(a * RN(1/c)) (kFast: c has no bits below bf16's and 2^-40 <= |c| <= 2^40; decided once per launch's
// uniform value, any other clamp value takes the division). clamp(rint(q), -128, 127) is sat_u8(rne(q + 128)) - 128:
// q is a bf16 number, so the sum is exact wherever it matters. A NaN becomes 0 (what the tensor library's
// float -> int8 conversion makes of it); the byte conversion would make it -128, so 8 inputs with a NaN among
// them take the slow form.
template <bool kFast>
__device__ __forceinline__ u32x2_t act_quant8(const u32x4_t v, float c, float r) {
    unsigned w[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float f = (j & 1) ? lq_bf16_hi(v[j >> 1]) : lq_bf16_lo(v[j >> 1]);
        const float a = lq_bf16r(f * 127.0f);
        if (kFast) {
            const float q = lq_bf16r(a * r) + 128.0f;
            switch (j & 3) {
                case 0: w[j >> 2] = act_cvt_pk_u8<0>(q, w[j >> 2]); break;
                case 1: w[j >> 2] = act_cvt_pk_u8<1>(q, w[j >> 2]); break;
                case 2: w[j >> 2] = act_cvt_pk_u8<2>(q, w[j >> 2]); break;
                default: w[j >> 2] = act_cvt_pk_u8<3>(q, w[j >> 2]); break;
            }
        } else {
            const float q = lq_bf16r(a / c);
            const float rr = q == q ? __builtin_amdgcn_fmed3f(rintf(q), -128.0f, 127.0f) : 0.0f;
            w[j >> 2] |= ((unsigned)(int)rr & 0xFFu) << (8 * (j & 3));
        }
    }
    if (kFast) return u32x2_t{w[0] ^ 0x80808080u, w[1] ^ 0x80808080u};
    return u32x2_t{w[0], w[1]};
}

// act_quant8 in the form the clamp value and the inputs allow (a NaN among the 8: the two forms differ on it, see above).
__device__ __forceinline__ u32x2_t act_quant8_any(const u32x4_t v, float c) {
    const bool c_is_bf16 = (__float_as_uint(c) & 0xFFFFu) == 0u && fabsf(c) >= 0x1p-40f && fabsf(c) <= 0x1p40f;
    bool any_nan = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) any_nan |= (v[j] & 0x7FFFu) > 0x7F80u || (v[j] & 0x7FFF0000u) > 0x7F800000u;
    return c_is_bf16 && !any_nan ? act_quant8<true>(v, c, 1.0f / c) : act_quant8<false>(v, c, 0.0f);
}

// 8 elements of a token row on the row's own scale: clamp(rint(x * inv), -128, 127), NaN -> 0
__device__ __forceinline__ u32x2_t act_quant8_token(const u32x4_t w, float inv) {
    unsigned o[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float f = (j & 1) ? lq_bf16_hi(w[j >> 1]) : lq_bf16_lo(w[j >> 1]);
        const float r = rintf(f * inv);
        const float rr = r == r ? __builtin_amdgcn_fmed3f(r, -128.0f, 127.0f) : 0.0f;
        o[j >> 2] |= ((unsigned)(int)rr & 0xFFu) << (8 * (j & 3));
    }
    return u32x2_t{o[0], o[1]};
}

// The larger of amax and the 8 magnitudes, as bf16 bit patterns
__device__ __forceinline__ unsigned act_amax8(const u32x4_t w, unsigned amax) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned a = w[j] & 0x7FFF7FFFu;
        const unsigned lo = a & 0xFFFFu, hi = a >> 16;
        amax = amax > lo ? amax : lo;
        amax = amax > hi ? amax : hi;
    }
    return amax;
}

// Order-preserving 16-bit key of a bf16 pattern: a larger value has a larger key, -0 < +0, and every NaN has the
// largest key of all, so that an integer maximum over the keys is the tensor library's max(), which returns NaN as
// soon as one element is NaN.
__device__ __forceinline__ unsigned max_key(unsigned b) {
    const unsigned a = b & 0x7FFFu;
    const unsigned k = (b & 0x8000u) ? 0x7FFFu - a : 0x8000u | a;
    return a > 0x7F80u ? 0xFFFFu : k;
}
__device__ __forceinline__ float max_key_value(unsigned k) {
    const unsigned b = k == 0xFFFFu ? 0x7FC0u : (k & 0x8000u) ? (k & 0x7FFFu) : 0x8000u | (0x7FFFu - k);
    return __uint_as_float(b << 16);
}

// The larger of k and the keys of 8 elements
__device__ __forceinline__ unsigned max_key8(const u32x4_t v, unsigned k) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned lo = max_key(v[j] & 0xFFFFu), hi = max_key(v[j] >> 16);
        k = k > lo ? k : lo;
        k = k > hi ? k : hi;
    }
    return k;
}

__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const unsigned other = (unsigned)__shfl_xor((int)v, o, 64);
        v = v > other ? v : other;
    }
    return v;
}
