// Forward of the A16W4 layers for 17 to 64 tokens and up to 16 columns per compute unit, in one launch:
//   Y[M,N] = X[M,K] . deq(W)[N,K]^T (+ bias)
//
// Bound: latency, and what a compute unit takes in from L2 (64 bytes a clock). The staged kernel (lq_gemm_staged.hip) has to cut K
// into slices to fill the device with such an output, and the launch that adds the slices costs as much as the product's
// own loop. Here a workgroup owns 16 columns and all of K, shared among its four waves: every compute unit reads all of X (0.5
// MB at 64 tokens and K = 4096: 3.9 us at that rate, the price of having no second launch).
//
// A wave takes every fourth group of 128 k and works on its own: its part of X, its codes, scales and zeros come by LDS-direct
// loads into stages that no other wave touches, D of them deep, with a wait and no barrier. The four partial sums meet in
// LDS at the end.
//
// us against the staged kernel with its second launch (and 16-token GEMV launches up to 32 tokens), weights from HBM:
//     N x K          17 tokens       32              48              64
//     4096 x 4096    10.3 -> 7.2     11.4 -> 7.6     13.6 -> 8.8     12.3 -> 9.9
//     2560 x 2560    9.9 -> 6.3      9.8 -> 6.3      10.0 -> 6.8     10.3 -> 7.4
//     4096 x 1024    9.9 -> 6.0      9.7 -> 6.2      8.0 -> 6.0      8.0 -> 6.1
//     2560 x 8192    12.1 -> 9.7     12.9 -> 10.8    14.3 -> 13.2    15.0 / 15.6
//     4096 x 11008   15.8 -> 14.9    15.7 / 17.2     17.5 / 21.7     18.2 / 25.6   (the last three stay with the staged kernel)
// (measured then; one load of scales for two groups: 4096 x 4096 at 17 / 32 / 45 / 64 tokens 7.70 / 9.06 / 10.44 / 12.09 -> 7.56 / 8.83 /
// 10.14 / 11.63 on another card)
// X arrives at 30 bytes a clock and unit, half of what L2 gives a unit reading alone; letting the units start at different
// groups changes nothing.
//
// Weights are not rounded to bf16, as they are not in the GEMV (lq_gemv.hip), which ran most of these sizes before: the operand
// is q - rint(z), exact in bf16, and the scale is applied in fp32 to the sum of a group.
//
// MFMA 16x16x32, activations first: lane l holds column l % 16 of tokens 4 (l / 16) .. + 3, so that the scale is one
// number. With r = l % 16, h = l / 16 slice w = 0..3 of a group has the lane's operands at k = 32 h + 8 w .. + 7: word w of
// the 16 bytes of codes of row r, and a 16-byte piece of X.
#include "lq_common.h"

#include <type_traits>

namespace {

struct FewParams {
    const unsigned char *x;  // bf16 [M, K]
    const unsigned char *w;  // packed codes
    const unsigned short *scales, *zeros, *bias;
    unsigned short *y;       // bf16 [M, N]
    int M, N, K;
    unsigned long long *clk; // measurement aid, see lq_calib_gemm_clocks; null in normal use
};

typedef __attribute__((address_space(3))) void lds_void;

template <int I>
using ic = std::integral_constant<int, I>;

constexpr int kWaves = 4;

// LDS layout of a wave's stage (16-byte pieces, swizzled so that 16 lanes reading one piece of 16 rows cover all banks):
//   activations  16 MT rows of 256 bytes, piece c of row i at c ^ (i & 15)
//   codes        16 rows of 64 bytes, piece c of row i at c ^ ((i >> 2) & 3)
// and beside the stages four slots of scales and zeros, one load for every two of the wave's groups (each 2-byte value pulls a
// cache line through L1, 32 of the 144 a group took with 48 tokens; the two groups' are 8 bytes apart):
//   dword 32 e + i: the scale, 32 e + 16 + i: the zero of row i for the first (e = 0) or second group, in the lower half
// MT: groups of 16 tokens, D: stages. Arguments: those of the first loads first (the leading 14 dwords are preloaded, build.py)
template <int MT, int D>
__global__ __launch_bounds__(64 * kWaves) void gemm_few_kernel(
    const unsigned char *x_, const unsigned char *w_, int M, int N, int K, const unsigned short *scales, const unsigned short *zeros,
    const unsigned short *bias, unsigned short *y, unsigned long long *clk) {
    const FewParams p = {x_, w_, scales, zeros, bias, y, M, N, K, clk};
    constexpr int A_BYTES = MT * 4096, STAGE = A_BYTES + 1024, WAVE = D * STAGE + 4 * 256;
    constexpr int LOADS = 4 * MT + 1;  // per stage; one more in the first of two
    static_assert((D - 1) * (LOADS + 1) < 64, "the wait counts loads in six bits");
    __shared__ __attribute__((aligned(16))) unsigned char lds[kWaves * WAVE];

    unsigned long long clk_t0 = 0, clk_r0 = 0;
    if (p.clk) {
        clk_t0 = __builtin_amdgcn_s_memtime();
        clk_r0 = __builtin_amdgcn_s_memrealtime();
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, h = lane >> 4;
    const int c0 = blockIdx.x * 16;
    const int G = p.K / LQ_GROUP;
    unsigned char *const mine = lds + wave * WAVE, *const q_ring = mine + D * STAGE;

    // ---- loads: instruction i < 4 MT brings rows 4 i .. 4 i + 3 of the wave's group of X
    const unsigned lda = (unsigned)p.K * 2u;
    unsigned a_off[4 * MT];
#pragma unroll
    for (int i = 0; i < 4 * MT; ++i) {
        const int row = 4 * i + (lane >> 4);
        a_off[i] = (unsigned)(row < p.M ? row : p.M - 1) * lda + ((lane & 15) ^ (row & 15)) * 16;
    }
    const int crow = lane >> 2;
    const unsigned c_off = (unsigned)crow * (unsigned)(p.K / 2) + ((lane & 3) ^ ((crow >> 2) & 3)) * 16;
    const unsigned q_off = (unsigned)r * (unsigned)G * 2u;
    const unsigned char *c_base = p.w + (long long)c0 * (p.K / 2);
    const unsigned char *s_base = (const unsigned char *)(p.scales + (long long)c0 * G);
    const unsigned char *z_base = (const unsigned char *)(p.zeros + (long long)c0 * G);
    // scales on lanes 0..15, zeros on 16..31, the next group's on 32..63: one instruction, 64-bit addresses
    const unsigned char *q_lane = (h & 1 ? z_base : s_base) + q_off;
    auto to_lds = [&](unsigned char *dst, unsigned off, const unsigned char *src) {
        const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)dst);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
    };
    const int ng = wave < G ? (G - wave + kWaves - 1) / kWaves : 0;  // the wave's groups: wave, wave + 4, ...
    auto group_at = [&](int i) { return wave + kWaves * (i < ng ? i : ng - 1); };
    // the wave's group i into stage st, the codes (from HBM) first; past the last group: that one again (nothing uses it)
    auto issue = [&](int i, unsigned char *st) {
        const int g = group_at(i);
        to_lds(st + A_BYTES, c_off, c_base + (long long)g * 64);
        if (!(i & 1)) {
            const unsigned q_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(q_ring + ((i >> 1) & 3) * 256));
            const int gq = h < 2 ? g : group_at(i + 1);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off" ::"s"(q_addr), "v"(q_lane + (long long)gq * 2) : "memory");
        }
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k) to_lds(st + k * 1024, a_off[k], p.x + (long long)g * 256);
    };

    f32x4_t acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    auto group = [&](int i, auto si) {
        constexpr int S = decltype(si)::value;
        unsigned char *st = mine + S * STAGE;
        // the D - 1 later stages' loads may be under way; how many of those are first ones of two follows from D and, where D is
        // even, the stage
        constexpr int FIRSTS = D == 3 ? 1 : D / 2 - 1 + (S & 1);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LOADS + FIRSTS) : "memory");
        const u32x4_t c = *reinterpret_cast<const u32x4_t *>(st + A_BYTES + r * 64 + ((h ^ ((r >> 2) & 3)) << 4));
        const unsigned *q = reinterpret_cast<const unsigned *>(q_ring + ((i >> 1) & 3) * 256) + 32 * (i & 1);
        const float sc = __uint_as_float(q[r] << 16);
        float zi, rest;
        lq_split_zero(__uint_as_float(q[16 + r] << 16), zi, rest);
        u32x4_t x[4][MT];
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int j = 0; j < MT; ++j) x[w][j] = *reinterpret_cast<const u32x4_t *>(st + (16 * j + r) * 256 + (((4 * h + w) ^ r) << 4));
        // the stage is free once these reads have returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue(i + D, st);
        __builtin_amdgcn_sched_barrier(0);
        f32x4_t P[MT];
#pragma unroll
        for (int j = 0; j < MT; ++j) P[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        auto add = [&](int w, const u32x4_t &b) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
                P[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[w][j]), __builtin_bit_cast(bf16x8_t, b), P[j], 0, 0, 0);
        };
#pragma unroll
        for (int w = 0; w < 4; ++w) add(w, lq_codes_minus(c[w], zi));
        if (__builtin_amdgcn_ballot_w64(rest != 0.0f)) {
            const u32x4_t b = lq_minus_rest(rest);
#pragma unroll
            for (int w = 0; w < 4; ++w) add(w, b);
        }
#pragma unroll
        for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][e] = fmaf(sc, P[j][e], acc[j][e]);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (ng > 0) {
#pragma unroll
        for (int d = 0; d < D; ++d) issue(d, mine + d * STAGE);
        int i = 0;
        for (; i + D <= ng; i += D) {
            group(i, ic<0>());
            group(i + 1, ic<1>());
            if constexpr (D > 2) group(i + 2, ic<2 % D>());
            if constexpr (D > 3) group(i + 3, ic<3 % D>());
        }
        static_assert(D >= 2 && D <= 4, "the loop above names up to four stages");
        if (i < ng) group(i, ic<0>());
        if constexpr (D > 2) if (i + 1 < ng) group(i + 1, ic<1>());
        if constexpr (D > 3) if (i + 2 < ng) group(i + 2, ic<2 % D>());
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped loads of the last groups
    __syncthreads();

    // ---- partial sums [wave][token][16 columns]
    float *part = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[((wave * MT + j) * 16 + 4 * h + e) * 16 + r] = acc[j][e];
    __syncthreads();
    for (int q = threadIdx.x; q < MT * 64; q += 64 * kWaves) {
        const int m = q >> 2, c = c0 + 4 * (q & 3);
        if (m >= p.M) continue;
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const f32x4_t a = *reinterpret_cast<const f32x4_t *>(part + w * (MT * 256) + q * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += a[e];
        }
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += lq_bf16_bits_to_f32(p.bias[c + e]);
        }
        *reinterpret_cast<u32x2_t *>(p.y + (long long)m * p.N + c) = u32x2_t{lq_pack_bf16(v[0], v[1]), lq_pack_bf16(v[2], v[3])};
    }
    if (p.clk && threadIdx.x == 0) {
        unsigned long long *c = p.clk + 4ll * blockIdx.x;
        c[0] = clk_t0; c[1] = __builtin_amdgcn_s_memtime(); c[2] = clk_r0; c[3] = __builtin_amdgcn_s_memrealtime();
    }
}

}  // namespace

// 16 < M <= 64, N % 16 == 0, K % 128 == 0 are guaranteed by the caller.
int lq_gemm_few_launch(const void *x, const void *codes, const void *scales, const void *zeros, const void *bias, void *y, int M, int N,
                       int K, hipStream_t st, unsigned long long *clk, const char *who) {
    FewParams p = {};
    p.x = (const unsigned char *)x; p.w = (const unsigned char *)codes;
    p.scales = (const unsigned short *)scales; p.zeros = (const unsigned short *)zeros;
    p.bias = (const unsigned short *)bias; p.y = (unsigned short *)y;
    p.M = M; p.N = N; p.K = K; p.clk = clk;
    // the 32-bit lane offsets of the loads span the tokens' rows and 16 rows of codes
    if (128ll * K >= (1ll << 32)) return lq_fail(LQ_ERR_BAD_ARG, "%s: K too large", who);
    const dim3 grid((unsigned)(N / 16)), block(64 * kWaves);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, p.x, p.w, M, N, K, p.scales, p.zeros, p.bias, p.y, clk); };
    if (M <= 32) launch(gemm_few_kernel<2, 4>);
    else if (M <= 48) launch(gemm_few_kernel<3, 3>);
    else launch(gemm_few_kernel<4, 2>);
    return lq_check_launch(who);
}
