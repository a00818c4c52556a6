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
// acc + (low or high 16 bits of word) * times, saturating at 2^32 - 1
template <int HI>
__device__ __forceinline__ unsigned add_half_sat(unsigned word, unsigned times, unsigned acc) {
    unsigned r;
    if (HI) asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0] clamp" : "=v"(r) : "v"(word), "s"(times), "v"(acc));
    else asm("v_mad_u32_u16 %0, %1, %2, %3 clamp" : "=v"(r) : "v"(word), "s"(times), "v"(acc));
    return r;
}

// The definition, one operation per line (any inputs). a < 65536.
__device__ __forceinline__ unsigned requant_elem(unsigned q, float s, float z, float g, float lr, unsigned a) {
    const float d = lq_bf16r((float)q - z);
    const float w = lq_bf16r(d * s);
    const float t = fmaf(-lr, g, w);
    const float r16 = (1.0f / s) * 65536.0f;
    const float c16 = fmaf(z, 65536.0f, 0.5f);
    const unsigned S = add_half_sat<0>(a, 1u, cvt_u32_sat(fmaf(t, r16, c16)));
    const unsigned c = S >> 16;
    return c > 15u ? 15u : c;
}

// Per-group constants of the one-fma form. It stands for the definition's two roundings when z is an integer with
// |z| <= 240 (q - z is then exact in bf16) and s is far from the ends of the range (2^28 / s is finite); elsewhere (fast = false) the
// elements go through requant_elem.
struct RequantGroup {
    float s512, nzs, r28, c28;  // r28, c28: y of the definition times 2^12
    bool fast;
};
__device__ __forceinline__ RequantGroup requant_group(float s, float z) {
    RequantGroup p;
    p.fast = (z == floorf(z)) && (fabsf(z) <= 240.0f) && (s >= 0x1p-99f) && (s <= 0x1p100f);
    p.r28 = (1.0f / s) * 0x1p28f;
    p.nzs = -(z * s);
    p.s512 = s * 512.0f;
    p.c28 = fmaf(z, 0x1p28f, 2048.0f);
    return p;
}

// One word (8 consecutive elements): codes cw, update directions gv, the four Philox words aw (one 16-bit draw per
// element), step lr. The one-fma form; the caller redoes the word with requant_elem where p.fast is false.
// All of the definition's fixed point times 2^12: floor((2^12 y + 2^12 a) / 2^28) is its floor((y + a) / 2^16) whatever lies below
// a whole y, both saturate where the code is 15, and the code then is a sum's top nibble, which one instruction appends to the
// word (with the code in byte 2 a clamp and a gather of bytes took two instructions an element: 8192 x 2048 10.54 -> 10.30 us, a decoder
// layer's optimizer step 83.1 -> 82.5).
__device__ __forceinline__ unsigned requant_word(unsigned cw, const float (&gv)[8], const unsigned (&aw)[4], float lr,
                                                 const RequantGroup &p) {
    const unsigned lo4 = cw & 0x0F0F0F0Fu;         // odd elements
    const unsigned hi4 = (cw >> 4) & 0x0F0F0F0Fu;  // even elements
    // the codes as q/512, two per conversion
    const lq_f32x2_t e0 = lq_nibbles_lo(hi4), e1 = lq_nibbles_hi(hi4), o0 = lq_nibbles_lo(lo4), o1 = lq_nibbles_hi(lo4);
    const float qf[8] = {e0[0], o0[0], e0[1], o0[1], e1[0], o1[0], e1[1], o1[1]};
    unsigned word = 0;
#pragma unroll
    for (int i = 7; i >= 0; --i) {
        const int j = i ^ 1;  // element j is nibble j ^ 1 of the word: the highest nibble first
        const float t = fmaf(-lr, gv[j], lq_bf16r(fmaf(qf[j], p.s512, p.nzs)));
        const unsigned X = cvt_u32_sat(fmaf(t, p.r28, p.c28));
        const unsigned S = (j & 1) ? add_half_sat<1>(aw[j >> 1], 4096u, X) : add_half_sat<0>(aw[j >> 1], 4096u, X);
        word = __builtin_amdgcn_alignbit(word, S, 28);  // (word << 4) | (S >> 28)
    }
    return word;
}

}  // namespace
