// Arithmetic of the stochastic-rounding requantizer, shared by the stand-alone pass (lq_requant.hip, which states the
// definition) and the optimizer step that ends in it (lq_adam8.hip).
#pragma once
#include "lq_common.h"

namespace {

// float -> uint32, truncating, saturating: NaN and negatives give 0, values >= 2^32 give 2^32 - 1
__device__ __forceinline__ unsigned cvt_u32_sat(float x) {
    unsigned r;
    asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
// acc + (low or high 16 bits of word), saturating at 2^32 - 1
template <int HI>
__device__ __forceinline__ unsigned add_half_sat(unsigned word, unsigned acc) {
    unsigned r;
    if (HI) asm("v_mad_u32_u16 %0, %1, 1, %2 op_sel:[1,0,0,0] clamp" : "=v"(r) : "v"(word), "v"(acc));
    else asm("v_mad_u32_u16 %0, %1, 1, %2 clamp" : "=v"(r) : "v"(word), "v"(acc));
    return r;
}

// The definition, one operation per line (any inputs). a < 65536.
__device__ __forceinline__ unsigned requant_elem(unsigned q, float s, float z, float g, float lr, unsigned a) {
    const float d = lq_bf16r((float)q - z);
    const float w = lq_bf16r(d * s);
    const float t = fmaf(-lr, g, w);
    const float r16 = (1.0f / s) * 65536.0f;
    const float c16 = fmaf(z, 65536.0f, 0.5f);
    const unsigned S = add_half_sat<0>(a, cvt_u32_sat(fmaf(t, r16, c16)));
    const unsigned c = S >> 16;
    return c > 15u ? 15u : c;
}

// Per-group constants of the one-fma form. It stands for the definition's two roundings when z is an integer with
// |z| <= 240 (q - z is then exact in bf16) and s is far from the ends of the range; elsewhere (fast = false) the
// elements go through requant_elem.
struct RequantGroup {
    float s512, nzs, r16, c16;
    bool fast;
};
__device__ __forceinline__ RequantGroup requant_group(float s, float z) {
    RequantGroup p;
    p.fast = (z == floorf(z)) && (fabsf(z) <= 240.0f) && (s >= 0x1p-100f) && (s <= 0x1p100f);
    p.r16 = (1.0f / s) * 65536.0f;
    p.nzs = -(z * s);
    p.s512 = s * 512.0f;
    p.c16 = fmaf(z, 65536.0f, 0.5f);
    return p;
}

// One word (8 consecutive elements): codes cw, update directions gv, the four Philox words aw (one 16-bit draw per
// element), step lr. The one-fma form; the caller redoes the word with requant_elem where p.fast is false.
__device__ __forceinline__ unsigned requant_word(unsigned cw, const float (&gv)[8], const unsigned (&aw)[4], float lr,
                                                 const RequantGroup &p) {
    const unsigned lo4 = cw & 0x0F0F0F0Fu;         // odd elements
    const unsigned hi4 = (cw >> 4) & 0x0F0F0F0Fu;  // even elements
    // the codes as q/512, two per conversion
    const lq_f32x2_t e0 = lq_nibbles_lo(hi4), e1 = lq_nibbles_hi(hi4), o0 = lq_nibbles_lo(lo4), o1 = lq_nibbles_hi(lo4);
    const float qf[8] = {e0[0], o0[0], e0[1], o0[1], e1[0], o1[0], e1[1], o1[1]};
    unsigned S[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float t = fmaf(-lr, gv[j], lq_bf16r(fmaf(qf[j], p.s512, p.nzs)));
        const unsigned X = cvt_u32_sat(fmaf(t, p.r16, p.c16));
        const unsigned Sj = (j & 1) ? add_half_sat<1>(aw[j >> 1], X) : add_half_sat<0>(aw[j >> 1], X);
        S[j] = Sj < 0xFFFFFu ? Sj : 0xFFFFFu;  // code <= 15
    }
    // code of element j = byte 2 of S[j]; even elements go to the high nibbles, odd ones to the low
    const unsigned sel = 0x0C0C0602u;  // bytes (S1.b2, S0.b2, 0, 0) of v_perm_b32(S0, S1)
    const unsigned ev = (__builtin_amdgcn_perm(S[6], S[4], sel) << 16) | __builtin_amdgcn_perm(S[2], S[0], sel);
    const unsigned od = (__builtin_amdgcn_perm(S[7], S[5], sel) << 16) | __builtin_amdgcn_perm(S[3], S[1], sel);
    return (ev << 4) | od;
}

}  // namespace
