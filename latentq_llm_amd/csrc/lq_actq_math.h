// Arithmetic of the activation quantisers: shared by the passes of lq_actq.hip and the kernel that quantises a few tokens
// on its way into an int8 product (lq_gemv_i8.hip).
#pragma once
#include "lq_common.h"

#include <type_traits>

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
// kOwnMax: c is the maximum of the tensor the 8 belong to, which a NaN among them would have made a NaN.
template <bool kOwnMax>
__device__ __forceinline__ u32x2_t act_quant8_any(const u32x4_t v, float c) {
    const bool c_is_bf16 = (__float_as_uint(c) & 0xFFFFu) == 0u && fabsf(c) >= 0x1p-40f && fabsf(c) <= 0x1p40f;
    bool any_nan = false;
    if constexpr (!kOwnMax) {
#pragma unroll
        for (int j = 0; j < 4; ++j) any_nan |= (v[j] & 0x7FFFu) > 0x7F80u || (v[j] & 0x7FFF0000u) > 0x7F800000u;
    }
    return c_is_bf16 && !any_nan ? act_quant8<true>(v, c, 1.0f / c) : act_quant8<false>(v, c, 0.0f);
}

// 8 elements of a token row on the row's own scale: clamp(rint(x * inv), -128, 127), NaN -> 0. `finite`: the row's largest
// |x| and inv are, so that no product is a NaN, and sat_u8(rint + 128) - 128 is the clamp (both sums exact where it decides).
__device__ __forceinline__ u32x2_t act_quant8_token(const u32x4_t w, float inv, bool finite) {
    unsigned o[2] = {0u, 0u};
    if (finite) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float q[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
                q[j] = rintf(((j & 1) ? lq_bf16_hi(w[2 * h + (j >> 1)]) : lq_bf16_lo(w[2 * h + (j >> 1)])) * inv) + 128.0f;
            o[h] = act_cvt_pk_u8<0>(q[0], o[h]);
            o[h] = act_cvt_pk_u8<1>(q[1], o[h]);
            o[h] = act_cvt_pk_u8<2>(q[2], o[h]);
            o[h] = act_cvt_pk_u8<3>(q[3], o[h]);
        }
        return u32x2_t{o[0] ^ 0x80808080u, o[1] ^ 0x80808080u};
    }
    asm volatile("; one element at a time");  // (keeps this side from being computed along with the other one)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float f = (j & 1) ? lq_bf16_hi(w[j >> 1]) : lq_bf16_lo(w[j >> 1]);
        const float r = rintf(f * inv);
        const float rr = r == r ? __builtin_amdgcn_fmed3f(r, -128.0f, 127.0f) : 0.0f;
        o[j >> 2] |= ((unsigned)(int)rr & 0xFFu) << (8 * (j & 3));
    }
    return u32x2_t{o[0], o[1]};
}

typedef short act_s16x2_t __attribute__((ext_vector_type(2)));
typedef unsigned short act_u16x2_t __attribute__((ext_vector_type(2)));

// The larger of amax and the magnitudes of 8 elements, as bf16 bit patterns, for even and odd elements
__device__ __forceinline__ act_u16x2_t act_amax8(const u32x4_t w, act_u16x2_t amax) {
#pragma unroll
    for (int j = 0; j < 4; ++j) amax = __builtin_elementwise_max(amax, __builtin_bit_cast(act_u16x2_t, w[j] & 0x7FFF7FFFu));
    return amax;
}
__device__ __forceinline__ unsigned act_amax_of(act_u16x2_t a) { return a[0] > a[1] ? a[0] : a[1]; }
// whether quotients of a row with this largest |x| cannot be NaN
__device__ __forceinline__ bool act_finite_row(float amax, float inv) { return amax <= 3.4028234e38f && inv <= 3.4028234e38f; }

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

// The largest key of many elements, two at a time: bf16 patterns as signed 16-bit integers of the same order (negative ones
// with their magnitude inverted), the largest and the smallest of them, for even and odd elements. NaNs are beyond infinity on
// either side. Four instructions a pair, where a key and a maximum for each element took 22.
struct MaxKeys {
    act_s16x2_t most = {-32768, -32768}, least = {32767, 32767};
    __device__ __forceinline__ void add8(const u32x4_t v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const unsigned pair = v[j];  // (a bit cast of the element itself would read the vector's first)
            const act_s16x2_t b = __builtin_bit_cast(act_s16x2_t, pair);
            const act_s16x2_t k = b ^ ((b >> 15) & (short)0x7FFF);
            most = __builtin_elementwise_max(most, k);
            least = __builtin_elementwise_min(least, k);
        }
    }
    __device__ __forceinline__ unsigned key() const {  // as max_key; 0, below every key, without elements
        const int hi = most[0] > most[1] ? most[0] : most[1], lo = least[0] < least[1] ? least[0] : least[1];
        return hi > 0x7F80 || lo < (short)0x807F ? 0xFFFFu : (unsigned)(hi + 0x8000);
    }
};

// The largest v of the wave's 64 lanes, on all of them: across lanes within the vector registers (a shuffle through LDS takes
// a hundred cycles each of six times)
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
    auto step = [&](auto ctrl) {
        const unsigned other = (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, decltype(ctrl)::value, 0xf, 0xf, false);
        v = v > other ? v : other;
    };
    step(std::integral_constant<int, 0x111>());  // row_shr:1
    step(std::integral_constant<int, 0x112>());  // row_shr:2
    step(std::integral_constant<int, 0x114>());  // row_shr:4
    step(std::integral_constant<int, 0x118>());  // row_shr:8: the last lane of 16 has their maximum
    step(std::integral_constant<int, 0x142>());  // row_bcast:15
    step(std::integral_constant<int, 0x143>());  // row_bcast:31
    return (unsigned)__builtin_amdgcn_readlane((int)v, 63);
}
