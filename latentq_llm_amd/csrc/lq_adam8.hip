// Fused Adam step on 8-bit block-wise moments for gfx950.
//
// The reference's optimizer (utils/quant.py:1081-1134 with Qfunc_8bit_opt / DeQfunc_8bit_opt,
// :22-41) keeps both moments as uint8 with one fp32 (scale, max) pair per block of 2048 (or 128)
// elements, the second one as sqrt(v) + eps, and runs one step as a chain of ~25 elementwise
// tensor operations per parameter:
//     m  = bf16(max1 - q1 * scale1)                      s2 = max2 - q2 * scale2,  v = bf16(s2 * s2)
//     m  = bf16(m * beta1);  m = bf16(m + (1 - beta1) * g)
//     v  = bf16(v * beta2);  v = bf16(v + (1 - beta2) * g * g)
//     d  = bf16(sqrt(v));    d = bf16(d + eps)
//     p  = bf16(p - step * (m / d))                      (or, for the stochastic-rounding
//                                                         requantizer, direction = bf16(m / d))
//     per block: max = max(x), scale = (max - min(x)) * (1/255) + 1e-10,
//                q = clamp(rint((max - x) / scale), 0, 255)        for x = m and for x = d
// Every tensor operation computes in fp32 and rounds its result to the tensor's type; an
// operation of the form a + alpha * b is a fused multiply-add inside the tensor library's
// kernels. This kernel is that chain in one pass with the same rounding points, so its results
// equal the chain's bit for bit.
//
// What becomes of the direction is the kernel's mode: it updates a bf16 parameter, is stored, is fed straight into the
// stochastic-rounding requantizer (lq_requant_math.h: the codes are rewritten and the direction never stored), or
// updates a latent weight kept as codes + residual words, rebuilt and re-quantised on the spot with the arithmetic of
// lq_latent_w4_* / lq_latent_w8_*.
//
// The kernel is bound by vector-ALU issue (the bytes alone would take half its time), so the split and the sequences
// below are chosen for instructions per element: a block of 2048 is 128 threads of two 8-element chunks (4 M elements
// still give 16 waves per compute unit, and the block reduction costs 16 elements instead of 8), rounding to bf16 is one
// conversion whose other half is zero, and the operands on which a short sequence would not be exact are looked for with
// the minima and maxima that the block reduction needs anyway, one branch per chunk. Measured on 8192 x 2048 with
// operands from HBM (bytes at the 5.05 TB/s of a large copy in brackets), against the form with 8 elements per thread,
// two rounding instructions, two barriers and the exact square root computed beside the short one:
//   parameter 42.5 -> 37.6 us (33.3), direction 39.3 -> 30.7 (26.6), direction + requantizer 48.2 -> 33.7 in one pass
//   (23.3), int4 + residual 63.0 -> 46.8 (26.7), int8 + residual 60.4 -> 46.6 (29.9).
// A block of 2048 has 256 codes at most for each moment, and what the step makes of a stored moment before the gradient
// comes in (dequantise, round, square, decay, round: 13 instructions for the two) depends on nothing but the code: the block's
// 128 threads form the 512 values once and an element looks its two up in LDS (random reads; with their
// bank conflicts LDS is busy for a third of the launch). One block to a workgroup, so that a look-up is a byte shifted and a
// read. (Launches of few blocks and of two numbers between: neither, see adam8_tables.) A decoder layer's six weights (50 M elements): stochastic
// rounding 91.9 -> 85.3 us, int4 + residual 141.9 -> 134.7; 64 M elements: int8 + residual 164.5 -> 155.7, bf16 151.8 -> 147.8. 57 vector instructions an element are left of 65 in
// the first, and the vector ALUs are busy all the time. The extrema across lanes in registers instead of shuffles through LDS,
// and no minimum of the second moments with an eps that hides their subnormals, 50 M elements: stochastic rounding 90 -> 84 us,
// int4 + residual 133 -> 125.7, int8 + residual 134 -> 127, bf16 128 -> 124.4.
#include "lq_adam8_tables.h"
#include "lq_latent_math.h"
#include "lq_requant_math.h"

#include <new>
#include <vector>

namespace {

struct Adam8Params {
    const u32x4_t *grad;     // bf16
    u32x4_t *param;          // bf16, updated in place
    u32x4_t *direction;      // bf16 m / d (or |m / d|)
    u32x2_t *state1, *state2;  // uint8 moments, updated in place
    float *scale1, *max1, *scale2, *max2;  // per block, updated in place
    long long n_blocks;
    float beta1, one_minus_beta1, beta2, one_minus_beta2, eps, neg_step;
    // latent and stochastic-rounding modes of a 4-bit layer: one code word per 8 elements, group scales and zeros
    const unsigned *codes_in;
    unsigned *codes, *residual;
    const unsigned short *wscales, *wzeros;  // per group of 128 elements
    CodecParams dequant_curve, quant_curve;
    // latent mode of an 8-bit-weight layer: int8 codes (8 per thread), one bf16 scale per row of K elements
    u32x2_t *codes8;
    const unsigned short *qscales;
    long long chunks_per_row;  // K / 8
    unsigned long long seed, offset;  // stochastic rounding: one Philox block per chunk
};

// Several parameters in one launch: workgroups first[i] .. first[i + 1] - 1 work on a[i]. A parameter of 4 M elements gives a
// compute unit four workgroups, which all load, compute and store at the same time, and a launch of its own: 14.0 us where a
// quarter of 16 M elements takes 9.4. A decoder layer's six weights (50 M elements): stochastic rounding 119.5 -> 92.6 us, int4 +
// residual 174.6 -> 143.5.
constexpr int kAdam8Batch = 8;
struct Adam8Batch {
    Adam8Params a[kAdam8Batch];
    unsigned first[kAdam8Batch + 1];
    int n;
};

// What the step does with m / d
enum {
    ADAM_PARAM = 0,   // bf16 parameter in place
    ADAM_DIR = 1,     // bf16(m / d) stored
    ADAM_SR = 2,      // stochastic-rounding requantizer on 4-bit codes
    ADAM_W4 = 3,      // 4-bit codes + residual words
    ADAM_W8 = 4,      // int8 codes + residual words
    ADAM_RATIO = 5,   // bf16(|m| / d) stored and nothing updated
};

__device__ __forceinline__ float min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float min2(float a, float b) {  // (fminf would first quiet operands of unknown origin)
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float max2(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float min3_abs(float a, float b, float c) {  // of |a|, |b| and c
    float r;
    asm("v_min3_f32 %0, |%1|, |%2|, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Minima and maxima over the wave's 64 lanes (or each row of 16): across lanes within the vector registers, where shuffles
// through LDS took six round trips and as many address computations again. A row's results are on all of its lanes, the
// wave's on lane 63.
// One block of assembly, since the waits that a register needs between its write and a read across lanes are not put inside
// or before it: three other instructions lie between, and two wait states in front.
#define LQ_ADAM8_ACROSS(ctrl)                                       \
    "v_min_f32_dpp %0, %0, %0 " ctrl " row_mask:0xf bank_mask:0xf\n\t"  \
    "v_max_f32_dpp %1, %1, %1 " ctrl " row_mask:0xf bank_mask:0xf\n\t"  \
    "v_min_f32_dpp %2, %2, %2 " ctrl " row_mask:0xf bank_mask:0xf\n\t"  \
    "v_max_f32_dpp %3, %3, %3 " ctrl " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ void row_extrema(float &lo1, float &hi1, float &lo2, float &hi2) {
    asm volatile("s_nop 1\n\t" LQ_ADAM8_ACROSS("row_ror:8") LQ_ADAM8_ACROSS("row_ror:4") LQ_ADAM8_ACROSS("row_ror:2") LQ_ADAM8_ACROSS("row_ror:1")
                 : "+v"(lo1), "+v"(hi1), "+v"(lo2), "+v"(hi2));
}
__device__ __forceinline__ void wave_extrema(float &lo1, float &hi1, float &lo2, float &hi2) {
    row_extrema(lo1, hi1, lo2, hi2);
    asm volatile("s_nop 1\n\t" LQ_ADAM8_ACROSS("row_bcast:15") LQ_ADAM8_ACROSS("row_bcast:31") : "+v"(lo1), "+v"(hi1), "+v"(lo2), "+v"(hi2));
}

// x[8] -> uint8 codes with the block's (scale, max); returns them packed, 8 bytes.
// The quotient (hi - x) / scale must be the correctly rounded one (a quotient one ulp off can fall on the other side of
// a rounding tie). The divisor is shared by the whole block: with its correctly rounded reciprocal r = RN(1 / scale) and
// what that leaves out, rl = (1 - r scale) r, q = t r + t rl is within one ulp of t / scale, and one residual correction
// of a quotient within one ulp returns RN(t / scale) exactly (Markstein's theorem; the residual is exact as long as it
// does not underflow, and a numerator below 2^-100 gives code 0 either way because scale >= 1e-10). A scale above 2^60
// (or NaN) takes the plain division.
__device__ __forceinline__ u32x2_t quantize8(const float (&x)[8], float scale, float hi, float r, float rl) {
    unsigned w[2] = {0u, 0u};
    float q[8];
    if (scale <= 0x1p60f) {
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float t = hi - x[k];
            const float q0 = fmaf(t, r, t * rl);
            q[k] = fmaf(fmaf(-q0, scale, t), r, q0);
        }
    } else {
        asm volatile("; plain division");  // (keeps this side from being computed along with the other one)
#pragma unroll
        for (int k = 0; k < 8; ++k) q[k] = (hi - x[k]) / scale;
    }
    // clamp(rint(q), 0, 255) and the byte insertion in one instruction (round to nearest even, saturating,
    // NaN -> 0 like fmaxf(NaN, 0))
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        w[h] = act_cvt_pk_u8<0>(q[4 * h], w[h]);
        w[h] = act_cvt_pk_u8<1>(q[4 * h + 1], w[h]);
        w[h] = act_cvt_pk_u8<2>(q[4 * h + 2], w[h]);
        w[h] = act_cvt_pk_u8<3>(q[4 * h + 3], w[h]);
    }
    return u32x2_t{w[0], w[1]};
}

// BS elements share one (scale, max) pair per moment: TPB threads of CH chunks of 8 elements, chunk c of thread t being
// elements 8 (c TPB + t) .. + 7 of the block, so that every access of a wave is contiguous. BPW blocks per workgroup.
// TABLES: the block's 512 values by code in LDS (see the top of the file), else computed for each element
template <int BS, int MODE, bool TABLES>
__global__ __launch_bounds__(TABLES ? 128 : 256) void adam8_kernel(Adam8Batch b) {
    int which = 0;
    for (int i = 1; i < b.n; ++i) which = blockIdx.x >= b.first[i] ? i : which;
    const Adam8Params &a = b.a[which];
    constexpr int CH = BS == 2048 ? 2 : 1, TPB = BS / 8 / CH, BPW = (TABLES ? 128 : 256) / TPB;
    __shared__ float red[4][4];
    __shared__ float vtab[16];  // latent modes: dequantised values of the 16 residual nibbles
    static_assert(!TABLES || TPB == 128, "a workgroup is one block");
    __shared__ float tabs[2][TABLES ? 256 : 1];
    if constexpr (MODE == ADAM_W4 || MODE == ADAM_W8) {
        lq_latent_fill_value_table(vtab, a.dequant_curve);
        if constexpr (!TABLES) __syncthreads();
    }
    const int t = threadIdx.x % TPB;
    long long blk = (long long)(blockIdx.x - b.first[which]) * BPW + threadIdx.x / TPB;
    const bool live = blk < a.n_blocks;
    if (!live) blk = 0;
    const long long first = blk * (BS / 8) + t;  // the thread's first chunk; the next ones are TPB further
    u32x4_t g4[CH], p4[CH];
    u32x2_t q1[CH], q2[CH], c8[CH];
    unsigned cword[CH], rword[CH];
    unsigned short wsb[CH], wzb[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const long long T = first + c * TPB;
        g4[c] = a.grad[T];
        q1[c] = a.state1[T];
        q2[c] = a.state2[T];
        if constexpr (MODE == ADAM_PARAM) p4[c] = a.param[T];
        if constexpr (MODE == ADAM_W4 || MODE == ADAM_SR) {
            cword[c] = a.codes_in[T];
            wsb[c] = a.wscales[T >> 4];
            wzb[c] = a.wzeros[T >> 4];
        }
        if constexpr (MODE == ADAM_W8) {
            c8[c] = a.codes8[T];
            wsb[c] = a.qscales[T / a.chunks_per_row];
        }
        if constexpr (MODE == ADAM_W4 || MODE == ADAM_W8) rword[c] = a.residual[T];
    }
    const float sc1 = a.scale1[blk], mx1 = a.max1[blk], sc2 = a.scale2[blk], mx2 = a.max2[blk];

    // what a code contributes to the new moments
    auto first_moment = [&](float q) { return lq_bf16r(lq_bf16r(mx1 - q * sc1) * a.beta1); };
    auto second_moment = [&](float q) {
        const float s2 = mx2 - q * sc2;
        return lq_bf16r(lq_bf16r(s2 * s2) * a.beta2);
    };
    if constexpr (TABLES) {
#pragma unroll
        for (int i = 0; i < 256 / TPB; ++i) {
            const int q = t + i * TPB;
            tabs[0][q] = first_moment((float)q);
            tabs[1][q] = second_moment((float)q);
        }
        __syncthreads();
    }

    float m[CH][8], d[CH][8];
    float lo1, hi1, lo2, hi2;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const long long T = first + c * TPB;
        float v[8], ratio[8];
        float g[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) g[k] = (k & 1) ? lq_bf16_hi(g4[c][k >> 1]) : lq_bf16_lo(g4[c][k >> 1]);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const unsigned b1 = (q1[c][k >> 2] >> (8 * (k & 3))) & 0xFFu, b2 = (q2[c][k >> 2] >> (8 * (k & 3))) & 0xFFu;
            const float mk = TABLES ? tabs[0][b1] : first_moment((float)b1);
            const float vk = TABLES ? tabs[1][b2] : second_moment((float)b2);
            m[c][k] = lq_bf16r(fmaf(a.one_minus_beta1, g[k], mk));
            v[k] = lq_bf16r(fmaf(a.one_minus_beta2 * g[k], g[k], vk));
            // bf16(sqrt(v)) of a bf16 v: the square root of a number with 8 significant bits never comes closer than
            // 2^-19 (relative) to the midpoint of two bf16 values, so the hardware's one-ulp square root rounds to the
            // same bf16 value as the correctly rounded one (checked for every bf16 input by the CPU tests)
            d[c][k] = lq_bf16r(lq_bf16r_trans(__builtin_amdgcn_sqrtf(v[k])) + a.eps);
            // m / d of two bf16 numbers: reciprocal and product. Where the fp32 quotient itself enters an update, one
            // residual correction makes it the IEEE one: the quotient of two 8-bit significands keeps a relative
            // distance of at least 2^-33 from every midpoint of two fp32 numbers, and the corrected value is within
            // 2^-45 of it (every significand pair and every one-ulp variant of the reciprocal is checked on the CPU).
            // Where only bf16(m / d) is used the product does: the quotient never comes closer than 2^-17 to the
            // midpoint of two bf16 values.
            const float r = __builtin_amdgcn_rcpf(d[c][k]);
            ratio[k] = m[c][k] * r;
            if constexpr (MODE == ADAM_PARAM || MODE == ADAM_W4 || MODE == ADAM_W8)
                ratio[k] = fmaf(fmaf(-ratio[k], d[c][k], m[c][k]), r, ratio[k]);
        }
        float clo1 = m[c][0], chi1 = m[c][0], clo2 = d[c][0], chi2 = d[c][0], mmin = fabsf(m[c][0]), vmin = 1.0f;
        if (c) { clo1 = lo1; chi1 = hi1; clo2 = lo2; chi2 = hi2; }
#pragma unroll
        for (int k = 0; k < 8; k += 2) {
            clo1 = min3(m[c][k], m[c][k + 1], clo1); chi1 = max3(m[c][k], m[c][k + 1], chi1);
            clo2 = min3(d[c][k], d[c][k + 1], clo2); chi2 = max3(d[c][k], d[c][k + 1], chi2);
            mmin = min3_abs(m[c][k], m[c][k + 1], mmin);
        }
        // an eps of 2^-38 and more swallows every root of a v below 2^-126, the exact one and what the hardware makes of it (at
        // most 2^-63, a quarter of eps's last place), and normal v have the right root
        if (!(a.eps >= 0x1p-38f)) {
            vmin = v[0];
#pragma unroll
            for (int k = 0; k < 8; k += 2) vmin = min3(v[k], v[k + 1], vmin);
        }
        // The short sequences hold for v >= 2^-100 (or eps >= 2^-38) and 2^-80 <= |m| <= 2^80, 2^-40 <= d <= 2^40 (no subnormal, no
        // underflowing residual, no overflow; NaN and infinity pass through them as through the plain ones). Chunks
        // with anything else, zeros among them, take the plain operations.
        const bool plain = !(vmin >= 0x1p-100f && mmin >= 0x1p-80f && fmaxf(fabsf(clo1), fabsf(chi1)) <= 0x1p80f &&
                             clo2 >= 0x1p-40f && chi2 <= 0x1p40f);
        if (plain) {
            asm volatile("; plain square roots and divisions");
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                d[c][k] = lq_bf16r(lq_bf16r_trans(__builtin_sqrtf(v[k])) + a.eps);
                ratio[k] = m[c][k] / d[c][k];
            }
            // the extrema again: the short root of a subnormal is none of the elements
            clo2 = c ? lo2 : d[c][0];
            chi2 = c ? hi2 : d[c][0];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                clo2 = fminf(clo2, d[c][k]);
                chi2 = fmaxf(chi2, d[c][k]);
            }
        }
        lo1 = clo1; hi1 = chi1; lo2 = clo2; hi2 = chi2;

        if constexpr (MODE == ADAM_W4) {
            const float ws = lq_bf16_bits_to_f32(wsb[c]), wz = lq_bf16_bits_to_f32(wzb[c]);
            float out[8], wq[8];
            lq_latent_weights(cword[c], ws, wz, lq_latent_one_fma(ws, wz), wq);
            const lq_latent_offsets rq = lq_latent_value_offsets(rword[c]);
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float p = lq_bf16r(lq_latent_value(wq[k], lq_latent_value_of(vtab, rq, k), ws));
                out[k] = lq_bf16r(fmaf(a.neg_step, ratio[k], p));
            }
            const float wr = 1.0f / ws;
            unsigned cnew, rnew;
            if ((ws >= 0x1p-40f) && (ws <= 0x1p40f)) lq_latent_requant8<true>(out, ws, wz, wr, a.quant_curve, cnew, rnew);
            else lq_latent_requant8<false>(out, ws, wz, wr, a.quant_curve, cnew, rnew);
            if (live) {
                a.codes[T] = cnew;
                a.residual[T] = rnew;
            }
        } else if constexpr (MODE == ADAM_W8) {
            const float ws = lq_bf16_bits_to_f32(wsb[c]);
            const lq_latent_offsets rq = lq_latent_value_offsets(rword[c]);
            float out[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float p = lq_bf16r(lq_latent_w8_value(c8[c][k >> 2] >> (8 * (k & 3)), lq_latent_value_of(vtab, rq, k), ws));
                out[k] = lq_bf16r(fmaf(a.neg_step, ratio[k], p));
            }
            const float wr = 1.0f / ws;
            u32x2_t cnew;
            unsigned rnew;
            if ((fabsf(ws) >= 0x1p-40f) && (fabsf(ws) <= 0x1p40f)) lq_latent_w8_requant8<true>(out, ws, wr, a.quant_curve, cnew, rnew);
            else lq_latent_w8_requant8<false>(out, ws, wr, a.quant_curve, cnew, rnew);
            if (live) {
                a.codes8[T] = cnew;
                a.residual[T] = rnew;
            }
        } else if constexpr (MODE == ADAM_SR) {
            const float ws = lq_bf16_bits_to_f32(wsb[c]), wz = lq_bf16_bits_to_f32(wzb[c]);
            const unsigned long long ctr = a.offset + (unsigned long long)T;
            const lq_u4 A = lq_philox4x32_10((unsigned)ctr, (unsigned)(ctr >> 32), 0u, 0u, (unsigned)a.seed, (unsigned)(a.seed >> 32));
            const unsigned aw[4] = {A.x, A.y, A.z, A.w};
            float dir[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) dir[k] = lq_bf16r(ratio[k]);
            const RequantGroup rg = requant_group(ws, wz);
            unsigned cnew = requant_word(cword[c], dir, aw, -a.neg_step, rg);
            if (!rg.fast) {
                asm volatile("; one operation at a time");
                cnew = 0;
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    cnew |= requant_elem(lq_code(cword[c], k), ws, wz, dir[k], -a.neg_step, (aw[k >> 1] >> (16 * (k & 1))) & 0xFFFFu)
                            << (4 * (k ^ 1));
            }
            if (live) a.codes[T] = cnew;
        } else {
            float out[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if constexpr (MODE == ADAM_PARAM) {
                    const float p = (k & 1) ? lq_bf16_hi(p4[c][k >> 1]) : lq_bf16_lo(p4[c][k >> 1]);
                    out[k] = fmaf(a.neg_step, ratio[k], p);
                } else {
                    out[k] = MODE == ADAM_RATIO ? fabsf(ratio[k]) : ratio[k];
                }
            }
            const u32x4_t o = {lq_pack_bf16(out[0], out[1]), lq_pack_bf16(out[2], out[3]), lq_pack_bf16(out[4], out[5]),
                               lq_pack_bf16(out[6], out[7])};
            if (live) {
                if constexpr (MODE == ADAM_PARAM) a.param[T] = o;
                else a.direction[T] = o;
            }
        }
    }
    if constexpr (MODE == ADAM_RATIO) return;

    // the moments back to uint8 with the block's new (scale, max): minima and maxima over the block's threads (a
    // 16-lane row of the wave, or two waves, through LDS)
    static_assert(TPB == 16 || TPB == 128, "a block is a row of lanes or two waves");
    if constexpr (TPB == 16) {
        row_extrema(lo1, hi1, lo2, hi2);
    } else {
        wave_extrema(lo1, hi1, lo2, hi2);
        if ((threadIdx.x & 63) == 63) *reinterpret_cast<f32x4_t *>(red[threadIdx.x >> 6]) = f32x4_t{lo1, hi1, lo2, hi2};
        __syncthreads();
        const int w = TABLES ? 0 : threadIdx.x >> 7 << 1;  // the block's first wave
        const f32x4_t w0 = *reinterpret_cast<const f32x4_t *>(red[w]), w1 = *reinterpret_cast<const f32x4_t *>(red[w + 1]);
        lo1 = min2(w0[0], w1[0]); hi1 = max2(w0[1], w1[1]);
        lo2 = min2(w0[2], w1[2]); hi2 = max2(w0[3], w1[3]);
    }
    const float inv255 = 1.0f / 255.0f;  // the tensor library divides by a scalar as a multiplication by its reciprocal
    const float ns1 = (hi1 - lo1) * inv255 + 1e-10f;
    const float ns2 = (hi2 - lo2) * inv255 + 1e-10f;
    const float r1 = 1.0f / ns1, r2 = 1.0f / ns2;
    const float rl1 = fmaf(-r1, ns1, 1.0f) * r1, rl2 = fmaf(-r2, ns2, 1.0f) * r2;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
        const u32x2_t n1 = quantize8(m[c], ns1, hi1, r1, rl1), n2 = quantize8(d[c], ns2, hi2, r2, rl2);
        if (live) {
            a.state1[first + c * TPB] = n1;
            a.state2[first + c * TPB] = n2;
        }
    }
    if (live && t == 0) {
        a.scale1[blk] = ns1; a.max1[blk] = hi1;
        a.scale2[blk] = ns2; a.max2[blk] = hi2;
    }
}

struct Adam8Item {
    Adam8Params a;
    int mode, block;
};

// Items of one mode and block size in one launch: as many as leave a grid that can be launched, their number to *taken
template <int BS, int MODE, bool TABLES>
int adam8_launch_batch(const char *who, const Adam8Item *const *items, int n, hipStream_t st, int *taken) {
    constexpr int kPerWg = BS == 128 ? 16 : TABLES ? 1 : 2;  // blocks per workgroup
    Adam8Batch b = {};
    unsigned long long wgs = 0;
    for (b.n = 0; b.n < n; ++b.n) {
        const unsigned long long mine = (unsigned long long)((items[b.n]->a.n_blocks + kPerWg - 1) / kPerWg);
        if (wgs + mine > 0x7FFFFFFFull) break;  // (one item alone fits: adam8_check)
        b.a[b.n] = items[b.n]->a;
        b.first[b.n] = (unsigned)wgs;
        wgs += mine;
    }
    b.first[b.n] = (unsigned)wgs;
    *taken = b.n;
    hipLaunchKernelGGL((adam8_kernel<BS, MODE, TABLES>), dim3((unsigned)wgs), dim3(TABLES ? 128 : 256), 0, st, b);
    return lq_check_launch(who);
}

// The items of one mode and block size, kAdam8Batch to a launch; with tables or without by adam8_tables. (Without them one block to
// a workgroup: 6.8 and 6.95 us for 0.6 and 1.6 M elements, stochastic rounding, where two take 5.6 and 7.6.)
template <int BS, int MODE>
int adam8_launch_items(const char *who, const Adam8Item *const *items, int n, hipStream_t st) {
    for (int i0 = 0, taken = 0; i0 < n; i0 += taken) {
        const int most = n - i0 < kAdam8Batch ? n - i0 : kAdam8Batch;
        long long blocks = 0;
        for (int i = 0; i < most; ++i) blocks += items[i0 + i]->a.n_blocks;
        const int rc = BS == 2048 && adam8_tables(blocks, lq_device_cu_count()) ? adam8_launch_batch<BS, MODE, BS == 2048>(who, items + i0, most, st, &taken)
                                                                       : adam8_launch_batch<BS, MODE, false>(who, items + i0, most, st, &taken);
        if (rc) return rc;
    }
    return LQ_OK;
}

template <int MODE>
int adam8_launch_mode(const char *who, const Adam8Item *const *items, int n, int block, hipStream_t st) {
    return block == 2048 ? adam8_launch_items<2048, MODE>(who, items, n, st) : adam8_launch_items<128, MODE>(who, items, n, st);
}

// One item now, or into the caller's queue
template <int MODE>
int adam8_launch(const char *who, Adam8Params &a, int64_t n, int block_elems, void *stream, void *queue = nullptr) {
    a.n_blocks = n / block_elems;
    const Adam8Item item = {a, MODE, block_elems};
    if (queue) {
        try {
            static_cast<std::vector<Adam8Item> *>(queue)->push_back(item);
        } catch (const std::bad_alloc &) {
            return lq_fail(LQ_ERR_LAUNCH, "%s: out of host memory", who);
        }
        return LQ_OK;
    }
    const Adam8Item *one = &item;
    return adam8_launch_mode<MODE>(who, &one, 1, block_elems, (hipStream_t)stream);
}

}  // namespace

static int adam8_check(const char *who, const void *grad, const void *state1, const void *state2, const void *scale1,
                       const void *max1, const void *scale2, const void *max2, int64_t n, int block_elems) {
    LQ_REQUIRE(grad && state1 && state2 && scale1 && max1 && scale2 && max2, "%s: null pointer argument", who);
    LQ_REQUIRE(block_elems == 2048 || block_elems == 128, "%s: block must be 2048 or 128 elements, got %d", who, block_elems);
    LQ_REQUIRE(n > 0 && n % block_elems == 0, "%s: n=%lld must be a positive multiple of the block (%d)", who, (long long)n,
               block_elems);
    LQ_REQUIRE(n / 8 / 256 < 0x7FFFFFFFll, "%s: tensor too large", who);
    LQ_REQUIRE(lq_aligned(grad, 16) && lq_aligned(state1, 8) && lq_aligned(state2, 8) && lq_aligned(scale1, 4) &&
                   lq_aligned(max1, 4) && lq_aligned(scale2, 4) && lq_aligned(max2, 4),
               "%s: grad must be 16-byte, the moments 8-byte aligned", who);
    return LQ_OK;
}

static void adam8_scalars(Adam8Params &a, double beta1, double beta2, double eps, double step_size) {
    // the optimizer computes its scalars in double precision and the tensor library's kernels take them as fp32
    a.beta1 = (float)beta1; a.one_minus_beta1 = (float)(1.0 - beta1);
    a.beta2 = (float)beta2; a.one_minus_beta2 = (float)(1.0 - beta2);
    a.eps = (float)eps; a.neg_step = (float)(-step_size);
}

extern "C" int lq_adam8_update(const void *grad, void *param_or_null, void *direction_or_null, uint8_t *state1,
                               uint8_t *state2, float *scale1, float *max1, float *scale2, float *max2, int64_t n,
                               int block_elems, double beta1, double beta2, double eps, double step_size, void *stream) {
    int rc = adam8_check("lq_adam8_update", grad, state1, state2, scale1, max1, scale2, max2, n, block_elems);
    if (rc) return rc;
    LQ_REQUIRE((param_or_null != nullptr) != (direction_or_null != nullptr),
               "lq_adam8_update: exactly one of param and direction must be given");
    LQ_REQUIRE((!param_or_null || lq_aligned(param_or_null, 16)) && (!direction_or_null || lq_aligned(direction_or_null, 16)),
               "lq_adam8_update: param and direction must be 16-byte aligned");
    Adam8Params a = {};
    a.grad = (const u32x4_t *)grad;
    a.param = (u32x4_t *)param_or_null;
    a.direction = (u32x4_t *)direction_or_null;
    a.state1 = (u32x2_t *)state1; a.state2 = (u32x2_t *)state2;
    a.scale1 = scale1; a.max1 = max1; a.scale2 = scale2; a.max2 = max2;
    adam8_scalars(a, beta1, beta2, eps, step_size);
    if (param_or_null) return adam8_launch<ADAM_PARAM>("lq_adam8_update", a, n, block_elems, stream);
    return adam8_launch<ADAM_DIR>("lq_adam8_update", a, n, block_elems, stream);
}

extern "C" int lq_adam8_latent_w4_step_queued(const void *grad, void *codes, int32_t *residual, const void *scales,
                                       const void *zeros, uint8_t *state1, uint8_t *state2, float *scale1, float *max1,
                                       float *scale2, float *max2, int64_t N, int64_t K, int group, int block_elems,
                                       int dk1, float db1, int dk2, float db2, int dk3, int qk1, float qb1, int qk2,
                                       float qb2, int qk3, double beta1, double beta2, double eps, double step_size,
                                       void *stream, void *queue_or_null) {
    LQ_REQUIRE(N > 0 && K > 0 && K % LQ_GROUP == 0, "lq_adam8_latent_w4_step: need N > 0, K a positive multiple of %d",
               LQ_GROUP);
    LQ_REQUIRE(group == LQ_GROUP, "lq_adam8_latent_w4_step: group must be %d", LQ_GROUP);
    const int64_t n = N * K;
    int rc = adam8_check("lq_adam8_latent_w4_step", grad, state1, state2, scale1, max1, scale2, max2, n, block_elems);
    if (rc) return rc;
    LQ_REQUIRE(codes && residual && scales && zeros, "lq_adam8_latent_w4_step: null pointer argument");
    LQ_REQUIRE(lq_aligned(codes, 4) && lq_aligned(residual, 4), "lq_adam8_latent_w4_step: codes and residual must be 4-byte aligned");
    LQ_REQUIRE(dk1 > 0 && dk2 > 0 && dk3 > 0 && db1 > 0.0f && db2 > db1 && db2 < 0.5f && qk1 > 0 && qk2 > 0 && qk3 > 0 &&
                   qb1 > 0.0f && qb2 > qb1 && qb2 < 0.5f,
               "lq_adam8_latent_w4_step: need k1,k2,k3 > 0 and 0 < b1 < b2 < 0.5 for both curves");
    Adam8Params a = {};
    a.grad = (const u32x4_t *)grad;
    a.state1 = (u32x2_t *)state1; a.state2 = (u32x2_t *)state2;
    a.scale1 = scale1; a.max1 = max1; a.scale2 = scale2; a.max2 = max2;
    a.codes_in = a.codes = (unsigned *)codes; a.residual = (unsigned *)residual;
    a.wscales = (const unsigned short *)scales; a.wzeros = (const unsigned short *)zeros;
    a.dequant_curve = lq_codec_dequant_params(dk1, db1, dk2, db2, dk3);
    a.quant_curve = lq_codec_quant_params(qk1, qb1, qk2, qb2, qk3);
    adam8_scalars(a, beta1, beta2, eps, step_size);
    return adam8_launch<ADAM_W4>("lq_adam8_latent_w4_step", a, n, block_elems, stream, queue_or_null);
}

extern "C" int lq_adam8_latent_w4_step(const void *grad, void *codes, int32_t *residual, const void *scales,
                                       const void *zeros, uint8_t *state1, uint8_t *state2, float *scale1, float *max1,
                                       float *scale2, float *max2, int64_t N, int64_t K, int group, int block_elems,
                                       int dk1, float db1, int dk2, float db2, int dk3, int qk1, float qb1, int qk2,
                                       float qb2, int qk3, double beta1, double beta2, double eps, double step_size,
                                       void *stream) {
    return lq_adam8_latent_w4_step_queued(grad, codes, residual, scales, zeros, state1, state2, scale1, max1, scale2,
                                          max2, N, K, group, block_elems, dk1, db1, dk2, db2, dk3, qk1, qb1, qk2, qb2,
                                          qk3, beta1, beta2, eps, step_size, stream, nullptr);
}

extern "C" int lq_adam8_latent_w8_step_queued(const void *grad, int8_t *codes, int32_t *residual, const void *qscales, uint8_t *state1,
                                       uint8_t *state2, float *scale1, float *max1, float *scale2, float *max2, int64_t N,
                                       int64_t K, int block_elems, int dk1, float db1, int dk2, float db2, int dk3, int qk1,
                                       float qb1, int qk2, float qb2, int qk3, double beta1, double beta2, double eps,
                                       double step_size, void *stream, void *queue_or_null) {
    LQ_REQUIRE(N > 0 && K > 0 && K % 8 == 0, "lq_adam8_latent_w8_step: need N > 0, K a positive multiple of 8");
    const int64_t n = N * K;
    int rc = adam8_check("lq_adam8_latent_w8_step", grad, state1, state2, scale1, max1, scale2, max2, n, block_elems);
    if (rc) return rc;
    LQ_REQUIRE(codes && residual && qscales, "lq_adam8_latent_w8_step: null pointer argument");
    LQ_REQUIRE(lq_aligned(codes, 8) && lq_aligned(residual, 4) && lq_aligned(qscales, 2),
               "lq_adam8_latent_w8_step: codes must be 8-byte, residual 4-byte aligned");
    LQ_REQUIRE(dk1 > 0 && dk2 > 0 && dk3 > 0 && db1 > 0.0f && db2 > db1 && db2 < 0.5f && qk1 > 0 && qk2 > 0 && qk3 > 0 &&
                   qb1 > 0.0f && qb2 > qb1 && qb2 < 0.5f,
               "lq_adam8_latent_w8_step: need k1,k2,k3 > 0 and 0 < b1 < b2 < 0.5 for both curves");
    Adam8Params a = {};
    a.grad = (const u32x4_t *)grad;
    a.state1 = (u32x2_t *)state1; a.state2 = (u32x2_t *)state2;
    a.scale1 = scale1; a.max1 = max1; a.scale2 = scale2; a.max2 = max2;
    a.codes8 = (u32x2_t *)codes; a.residual = (unsigned *)residual;
    a.qscales = (const unsigned short *)qscales;
    a.chunks_per_row = K / 8;
    a.dequant_curve = lq_codec_dequant_params(dk1, db1, dk2, db2, dk3);
    a.quant_curve = lq_codec_quant_params(qk1, qb1, qk2, qb2, qk3);
    adam8_scalars(a, beta1, beta2, eps, step_size);
    return adam8_launch<ADAM_W8>("lq_adam8_latent_w8_step", a, n, block_elems, stream, queue_or_null);
}

extern "C" int lq_adam8_latent_w8_step(const void *grad, int8_t *codes, int32_t *residual, const void *qscales, uint8_t *state1,
                                       uint8_t *state2, float *scale1, float *max1, float *scale2, float *max2, int64_t N,
                                       int64_t K, int block_elems, int dk1, float db1, int dk2, float db2, int dk3, int qk1,
                                       float qb1, int qk2, float qb2, int qk3, double beta1, double beta2, double eps,
                                       double step_size, void *stream) {
    return lq_adam8_latent_w8_step_queued(grad, codes, residual, qscales, state1, state2, scale1, max1, scale2, max2,
                                          N, K, block_elems, dk1, db1, dk2, db2, dk3, qk1, qb1, qk2, qb2, qk3, beta1,
                                          beta2, eps, step_size, stream, nullptr);
}

extern "C" int lq_adam8_sr_step_queued(const void *grad, const void *codes_in, void *codes_out, const void *scales, const void *zeros,
                                uint8_t *state1, uint8_t *state2, float *scale1, float *max1, float *scale2, float *max2,
                                int64_t N, int64_t K, int group, int block_elems, double beta1, double beta2, double eps,
                                double step_size, uint64_t philox_seed, uint64_t philox_offset, void *stream, void *queue_or_null) {
    LQ_REQUIRE(N > 0 && K > 0 && K % LQ_GROUP == 0, "lq_adam8_sr_step: need N > 0, K a positive multiple of %d", LQ_GROUP);
    LQ_REQUIRE(group == LQ_GROUP, "lq_adam8_sr_step: group must be %d", LQ_GROUP);
    const int64_t n = N * K;
    int rc = adam8_check("lq_adam8_sr_step", grad, state1, state2, scale1, max1, scale2, max2, n, block_elems);
    if (rc) return rc;
    LQ_REQUIRE(codes_in && codes_out && scales && zeros, "lq_adam8_sr_step: null pointer argument");
    LQ_REQUIRE(lq_aligned(codes_in, 4) && lq_aligned(codes_out, 4) && lq_aligned(scales, 2) && lq_aligned(zeros, 2),
               "lq_adam8_sr_step: codes must be 4-byte, scales and zeros 2-byte aligned");
    Adam8Params a = {};
    a.grad = (const u32x4_t *)grad;
    a.state1 = (u32x2_t *)state1; a.state2 = (u32x2_t *)state2;
    a.scale1 = scale1; a.max1 = max1; a.scale2 = scale2; a.max2 = max2;
    a.codes_in = (const unsigned *)codes_in; a.codes = (unsigned *)codes_out;
    a.wscales = (const unsigned short *)scales; a.wzeros = (const unsigned short *)zeros;
    a.seed = philox_seed; a.offset = philox_offset;
    adam8_scalars(a, beta1, beta2, eps, step_size);
    return adam8_launch<ADAM_SR>("lq_adam8_sr_step", a, n, block_elems, stream, queue_or_null);
}

extern "C" int lq_adam8_sr_step(const void *grad, const void *codes_in, void *codes_out, const void *scales, const void *zeros,
                                uint8_t *state1, uint8_t *state2, float *scale1, float *max1, float *scale2, float *max2,
                                int64_t N, int64_t K, int group, int block_elems, double beta1, double beta2, double eps,
                                double step_size, uint64_t philox_seed, uint64_t philox_offset, void *stream) {
    return lq_adam8_sr_step_queued(grad, codes_in, codes_out, scales, zeros, state1, state2, scale1, max1, scale2,
                                   max2, N, K, group, block_elems, beta1, beta2, eps, step_size, philox_seed,
                                   philox_offset, stream, nullptr);
}

extern "C" int lq_adam8_queue_new(void **queue_out) {
    LQ_REQUIRE(queue_out, "lq_adam8_queue_new: null pointer argument");
    *queue_out = new (std::nothrow) std::vector<Adam8Item>;
    return *queue_out ? LQ_OK : lq_fail(LQ_ERR_LAUNCH, "lq_adam8_queue_new: out of host memory");
}

extern "C" int lq_adam8_queue_free(void *queue) {
    delete static_cast<std::vector<Adam8Item> *>(queue);
    return LQ_OK;
}

extern "C" int lq_adam8_queue_run(void *queue, void *stream) {
    LQ_REQUIRE(queue, "lq_adam8_queue_run: null pointer argument");
    std::vector<Adam8Item> items;
    items.swap(*static_cast<std::vector<Adam8Item> *>(queue));
    std::vector<const Adam8Item *> group;
    try {
        group.reserve(items.size());
    } catch (const std::bad_alloc &) {
        return lq_fail(LQ_ERR_LAUNCH, "lq_adam8_queue_run: out of host memory");
    }
    for (int mode : {ADAM_SR, ADAM_W4, ADAM_W8})
        for (int block : {2048, 128}) {
            group.clear();
            for (const Adam8Item &it : items)
                if (it.mode == mode && it.block == block) group.push_back(&it);
            if (group.empty()) continue;
            const char *who = "lq_adam8_queue_run";
            const int n = (int)group.size();
            hipStream_t st = (hipStream_t)stream;
            const int rc = mode == ADAM_SR ? adam8_launch_mode<ADAM_SR>(who, group.data(), n, block, st)
                           : mode == ADAM_W4 ? adam8_launch_mode<ADAM_W4>(who, group.data(), n, block, st)
                                             : adam8_launch_mode<ADAM_W8>(who, group.data(), n, block, st);
            if (rc) return rc;
        }
    return LQ_OK;
}

extern "C" int lq_adam8_ratio(const void *grad, const uint8_t *state1, const uint8_t *state2, const float *scale1,
                              const float *max1, const float *scale2, const float *max2, void *ratio_out, int64_t n,
                              int block_elems, double beta1, double beta2, double eps, void *stream) {
    int rc = adam8_check("lq_adam8_ratio", grad, state1, state2, scale1, max1, scale2, max2, n, block_elems);
    if (rc) return rc;
    LQ_REQUIRE(ratio_out && lq_aligned(ratio_out, 16), "lq_adam8_ratio: ratio_out must be given and 16-byte aligned");
    Adam8Params a = {};
    a.grad = (const u32x4_t *)grad;
    a.direction = (u32x4_t *)ratio_out;
    a.state1 = (u32x2_t *)state1; a.state2 = (u32x2_t *)state2;  // (read only in this mode)
    a.scale1 = (float *)scale1; a.max1 = (float *)max1; a.scale2 = (float *)scale2; a.max2 = (float *)max2;
    adam8_scalars(a, beta1, beta2, eps, 0.0);
    return adam8_launch<ADAM_RATIO>("lq_adam8_ratio", a, n, block_elems, stream);
}
