// Forward of the A16W4 layers for 17 to 128 tokens and up to 16 columns per compute unit, in one launch:
//   Y[M,N] = X[M,K] . deq(W)[N,K]^T (+ bias)
//
// Bound: latency, of the weights from HBM once and of X from L2 in rounds. The staged kernel (lq_gemm_staged.hip) has to cut K into
// slices to fill the device with such an output, and the launch that adds the slices costs as much as the product's own loop. Here a
// workgroup owns 16 columns and all of K, shared among its waves: every compute unit reads all of X (0.5 MB at 64 tokens and
// K = 4096, the price of having no second launch).
//
// A wave takes every W-th group of 128 k and works on its own, with waits and no barriers. All of its codes, scales and zeros are
// requested before anything else, into LDS that no other wave touches: 36 KB a workgroup at K = 4096. Loads return in order, so that
// codes requested among the rows of X, a few groups ahead, made every round of X wait for HBM. The rows of one group follow, are read into
// registers, and make place for the next group's while they are multiplied. The partial sums meet in LDS at the end. As many waves as
// LDS holds codes and one group of X for: two to a SIMD fill each other's waits, but codes ahead are worth more (a ring of six groups on
// eight waves 12 % slower at K = 5504 than all of them on six).
//
// us, codes three stages ahead on four waves -> all of them up front (both with weights from HBM):
//     N x K          17 tokens        32               45               64
//     4096 x 4096    7.75 -> 7.05     8.98 -> 7.72     10.3 -> 8.65     11.9 -> 9.8
//     2560 x 2560    5.65 -> 4.65     5.95 -> 4.72     6.87 -> 5.42     7.47 -> 6.44
//     4096 x 1024    4.38 -> 3.72     4.73 -> 3.79     5.20 -> 4.28     5.55 -> 4.88
//     2304 x 6144    9.56 -> 8.23     11.3 -> 8.42     13.3 -> 10.2     13.5 -> 11.6
//     4096 x 8192    13.5 -> 10.9     13.9 -> 11.0     16.1 -> 13.1     16.9 -> 15.8
// against the kernels of other sizes (GEMV launches up to 32 tokens, staged):
//     2048 x 4096    8.3 -> 5.8       9.4 -> 5.9       10.3 -> 6.9      10.8 -> 7.9
//     1536 x 1536                                      8.0 -> 4.5       8.2 -> 5.3
// From 65 tokens on and on long rows (rows of X in halves of a group, gemm_few_half_kernel), against the staged kernel's slices and the launch that adds them:
//                    65 tokens        80              96              128
//     4096 x 4096    12.6 -> 10.0                     13.5 -> 11.5    15.1 -> 13.9
//     1536 x 1536                     8.0 -> 5.6
//     2560 x 2560                                     11.3 -> 9.4 (97)
//     4096 x 9728 at 20 / 32 / 48 tokens 14.6 -> 12.9, 15.1 -> 13.0, 17.8 -> 15.4;  3072 x 9216 at 45 16.4 -> 13.3
// Also measured, 4096 x 4096 at 45 tokens: 32 columns a workgroup on half of the units 12.4; no rows of X after the first group 7.2, of
// the weights 8.0; no conversions 8.5, no LDS reads 8.6; units starting at different groups 8.8; codes of neighbouring groups in one
// piece of 128 bytes 8.7; X requested ahead of all but the first group's codes 8.6 (2560 x 2560 5.8).
//
// Weights are not rounded to bf16, as they are not in the GEMV (lq_gemv.hip), which ran most of these sizes before: the operand
// is q - rint(z), exact in bf16, and the scale is applied in fp32 to the sum of a group.
//
// MFMA 16x16x32, activations first: lane l holds column l % 16 of tokens 4 (l / 16) .. + 3, so that the scale is one
// number. With r = l % 16, h = l / 16 slice w = 0..3 of a group has the lane's operands at k = 32 h + 8 w .. + 7: word w of
// the 16 bytes of codes of row r, and a 16-byte piece of X.
#include "lq_common.h"

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

__device__ __forceinline__ void few_to_lds(unsigned char *dst, unsigned off, const unsigned char *src) {
    const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)dst);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
}

// The codes, scales and zeros of 16 columns
struct FewColumns {
    const unsigned char *c_base, *q_lane;
    unsigned c_off;
    int h;
    __device__ __forceinline__ FewColumns(const FewParams &p, int c0, int G, int lane) : h(lane >> 4) {
        const int crow = lane >> 2;
        c_off = (unsigned)crow * (unsigned)(p.K / 2) + ((lane & 3) ^ ((crow >> 2) & 3)) * 16;
        c_base = p.w + (long long)c0 * (p.K / 2);
        // scales on lanes 0..15, zeros on 16..31, the next group's on 32..63: one instruction, 64-bit addresses
        q_lane = (const unsigned char *)((h & 1 ? p.zeros : p.scales) + (long long)c0 * G) + (unsigned)(lane & 15) * (unsigned)G * 2u;
    }
    template <int NG, class GroupAt>
    __device__ __forceinline__ void issue(unsigned char *codes, unsigned char *q, int ng, GroupAt &&group_at) const {
#pragma unroll
        for (int i = 0; i < NG; ++i)
            if (i < ng) {
                few_to_lds(codes + i * 1024, c_off, c_base + (long long)group_at(i) * 64);
                if (!(i & 1)) {
                    const unsigned q_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(q + (i >> 1) * 256));
                    const int gq = h < 2 ? group_at(i) : group_at(i + 1);
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, off" ::"s"(q_addr), "v"(q_lane + (long long)gq * 2) : "memory");
                }
            }
    }
};

// The waves' sums of 16 MT tokens and 16 columns meet in LDS and leave as bf16
template <int MT, int W>
__device__ __forceinline__ void few_finish(const FewParams &p, float *part, const f32x4_t (&acc)[MT], int c0, int wave, int r, int h) {
    // ---- partial sums [wave][token][16 columns]
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[((wave * MT + j) * 16 + 4 * h + e) * 16 + r] = acc[j][e];
    __syncthreads();
    for (int i = threadIdx.x; i < MT * 64; i += 64 * W) {
        const int m = i >> 2, c = c0 + 4 * (i & 3);
        if (m >= p.M) continue;
        f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const f32x4_t a = *reinterpret_cast<const f32x4_t *>(part + w * (MT * 256) + i * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += a[e];
        }
        if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += lq_bf16_bits_to_f32(p.bias[c + e]);
        }
        *reinterpret_cast<u32x2_t *>(p.y + (long long)m * p.N + c) = u32x2_t{lq_pack_bf16(v[0], v[1]), lq_pack_bf16(v[2], v[3])};
    }
}

// LDS of a wave (16-byte pieces, swizzled so that 16 lanes reading one piece of 16 rows cover all banks):
//   codes        NG groups, of 16 rows of 64 bytes, piece c of row i at c ^ ((i >> 2) & 3)
//   scales and zeros  256 bytes for two groups, one load (each 2-byte value pulls a cache line through L1):
//                dword 32 e + i: the scale, 32 e + 16 + i: the zero of row i for the first (e = 0) or second group, in the lower half
//   activations  16 MT rows of 256 bytes, piece c of row i at c ^ (i & 15)
constexpr int few_lds(int MT, int NG, int W) { return W * (NG * 1024 + (NG + 1) / 2 * 256 + MT * 4096); }

// MT: groups of 16 tokens, W: waves, NG: groups of 128 k a wave has room for. Arguments: those of the first loads first (the leading 14
// dwords are preloaded, build.py)
template <int MT, int NG, int W>
__global__ __launch_bounds__(64 * W) void gemm_few_kernel(
    const unsigned char *x_, const unsigned char *w_, int M, int N, int K, const unsigned short *scales, const unsigned short *zeros,
    const unsigned short *bias, unsigned short *y, unsigned long long *clk) {
    const FewParams p = {x_, w_, scales, zeros, bias, y, M, N, K, clk};
    constexpr int Q_AT = NG * 1024, X_AT = Q_AT + (NG + 1) / 2 * 256, WAVE = X_AT + MT * 4096;
    static_assert(W * WAVE == few_lds(MT, NG, W) && W * WAVE <= 160 << 10, "LDS");
    __shared__ __attribute__((aligned(16))) unsigned char lds[W * WAVE];

    unsigned long long clk_t0 = 0, clk_r0 = 0;
    if (p.clk) {
        clk_t0 = __builtin_amdgcn_s_memtime();
        clk_r0 = __builtin_amdgcn_s_memrealtime();
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, h = lane >> 4;
    const int c0 = blockIdx.x * 16;
    const int G = p.K / LQ_GROUP;
    unsigned char *const codes = lds + wave * WAVE, *const q = codes + Q_AT, *const rows = codes + X_AT;

    // ---- loads
    const FewColumns cols(p, c0, G, lane);
    const int ng = wave < G ? (G - wave + W - 1) / W : 0;  // the wave's groups: wave, wave + W, ...
    auto group_at = [&](int i) { return wave + W * (i < ng ? i : ng - 1); };
    // instruction i brings rows 4 i .. 4 i + 3 of the group; past the wave's last group: that one again (nothing uses it)
    const unsigned lda = (unsigned)p.K * 2u;
    unsigned a_off[4 * MT];
    auto issue_rows = [&](int i) {
        const int g = group_at(i);
#pragma unroll
        for (int k = 0; k < 4 * MT; ++k) few_to_lds(rows + k * 1024, a_off[k], p.x + (long long)g * 256);
    };

    f32x4_t acc[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    if (ng > 0) {
        cols.issue<NG>(codes, q, ng, group_at);
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) {
            const int row = 4 * i + (lane >> 4);
            a_off[i] = (unsigned)(row < p.M ? row : p.M - 1) * lda + ((lane & 15) ^ (row & 15)) * 16;
        }
        issue_rows(0);
    }
    for (int i = 0; i < ng; ++i) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const u32x4_t c = *reinterpret_cast<const u32x4_t *>(codes + i * 1024 + r * 64 + ((h ^ ((r >> 2) & 3)) << 4));
        const unsigned *qi = reinterpret_cast<const unsigned *>(q + (i >> 1) * 256) + 32 * (i & 1);
        const float sc = __uint_as_float(qi[r] << 16);
        float zi, rest;
        lq_split_zero(__uint_as_float(qi[16 + r] << 16), zi, rest);
        u32x4_t x[4][MT];
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int j = 0; j < MT; ++j) x[w][j] = *reinterpret_cast<const u32x4_t *>(rows + (16 * j + r) * 256 + (((4 * h + w) ^ r) << 4));
        // the rows' place is free once these reads have returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue_rows(i + 1);
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
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the rows behind the last group's
    __syncthreads();

    few_finish<MT, W>(p, reinterpret_cast<float *>(lds), acc, c0, wave, r, h);
    if (p.clk && threadIdx.x == 0) {
        unsigned long long *c = p.clk + 4ll * blockIdx.x;
        c[0] = clk_t0; c[1] = __builtin_amdgcn_s_memtime(); c[2] = clk_r0; c[3] = __builtin_amdgcn_s_memrealtime();
    }
}

// The same for 65 to 128 tokens and for long rows, where rows of X of a whole group would leave LDS room for few waves: they come 64 k at
// a time, and the sums of a group are scaled after both halves. LDS of a wave: codes, scales and zeros as above;
//   activations  16 MT rows of 128 bytes, piece c of row i at c ^ ((i >> 1) & 7)
// With r, h as above slice w = 0, 1 of half s has the lane's operands at k = 64 s + 16 h + 8 w .. + 7.
constexpr int few_half_lds(int MT, int NG, int W) { return W * (NG * 1024 + (NG + 1) / 2 * 256 + MT * 2048); }

template <int MT, int NG, int W>
__global__ __launch_bounds__(64 * W) void gemm_few_half_kernel(
    const unsigned char *x_, const unsigned char *w_, int M, int N, int K, const unsigned short *scales, const unsigned short *zeros,
    const unsigned short *bias, unsigned short *y, unsigned long long *clk) {
    const FewParams p = {x_, w_, scales, zeros, bias, y, M, N, K, clk};
    constexpr int Q_AT = NG * 1024, X_AT = Q_AT + (NG + 1) / 2 * 256, WAVE = X_AT + MT * 2048;
    static_assert(W * WAVE == few_half_lds(MT, NG, W) && W * WAVE <= 160 << 10 && MT * 1024 <= WAVE, "LDS");
    __shared__ __attribute__((aligned(16))) unsigned char lds[W * WAVE];

    unsigned long long clk_t0 = 0, clk_r0 = 0;
    if (p.clk) {
        clk_t0 = __builtin_amdgcn_s_memtime();
        clk_r0 = __builtin_amdgcn_s_memrealtime();
    }
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, h = lane >> 4;
    const int c0 = blockIdx.x * 16;
    const int G = p.K / LQ_GROUP;
    unsigned char *const codes = lds + wave * WAVE, *const q = codes + Q_AT, *const rows = codes + X_AT;
    const FewColumns cols(p, c0, G, lane);
    const int ng = wave < G ? (G - wave + W - 1) / W : 0;  // the wave's groups: wave, wave + W, ...
    auto group_at = [&](int i) { return wave + W * (i < ng ? i : ng - 1); };
    // step t is half t & 1 of group t / 2; instruction i brings rows 8 i .. 8 i + 7; past the wave's last group: that one again
    const unsigned lda = (unsigned)p.K * 2u;
    unsigned a_off[2 * MT];
    auto issue_rows = [&](int t) {
        const unsigned char *src = p.x + (long long)group_at(t >> 1) * 256 + (t & 1) * 128;
#pragma unroll
        for (int k = 0; k < 2 * MT; ++k) few_to_lds(rows + k * 1024, a_off[k], src);
    };

    f32x4_t acc[MT], P[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[j] = P[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    if (ng > 0) {
        cols.issue<NG>(codes, q, ng, group_at);
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) {
            const int row = 8 * i + (lane >> 3);
            a_off[i] = (unsigned)(row < p.M ? row : p.M - 1) * lda + ((lane & 7) ^ ((row >> 1) & 7)) * 16;
        }
        issue_rows(0);
    }
    for (int t = 0; t < 2 * ng; ++t) {
        const int i = t >> 1, s = t & 1;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const u32x2_t c = *reinterpret_cast<const u32x2_t *>(codes + i * 1024 + r * 64 + (((2 * s + (h >> 1)) ^ ((r >> 2) & 3)) << 4) + 8 * (h & 1));
        const unsigned *qi = reinterpret_cast<const unsigned *>(q + (i >> 1) * 256) + 32 * (i & 1);
        const float sc = __uint_as_float(qi[r] << 16);
        float zi, rest;
        lq_split_zero(__uint_as_float(qi[16 + r] << 16), zi, rest);
        u32x4_t x[2][MT];
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int j = 0; j < MT; ++j) x[w][j] = *reinterpret_cast<const u32x4_t *>(rows + (16 * j + r) * 128 + (((2 * h + w) ^ ((r >> 1) & 7)) << 4));
        // the rows' place is free once these reads have returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        issue_rows(t + 1);
        __builtin_amdgcn_sched_barrier(0);
        auto add = [&](int w, const u32x4_t &b) {
#pragma unroll
            for (int j = 0; j < MT; ++j)
                P[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, x[w][j]), __builtin_bit_cast(bf16x8_t, b), P[j], 0, 0, 0);
        };
#pragma unroll
        for (int w = 0; w < 2; ++w) add(w, lq_codes_minus(c[w], zi));
        if (__builtin_amdgcn_ballot_w64(rest != 0.0f)) {
            const u32x4_t b = lq_minus_rest(rest);
#pragma unroll
            for (int w = 0; w < 2; ++w) add(w, b);
        }
        if (s) {
#pragma unroll
            for (int j = 0; j < MT; ++j) {
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[j][e] = fmaf(sc, P[j][e], acc[j][e]);
                P[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the rows behind the last group's
    __syncthreads();
    few_finish<MT, W>(p, reinterpret_cast<float *>(lds), acc, c0, wave, r, h);
    if (p.clk && threadIdx.x == 0) {
        unsigned long long *c = p.clk + 4ll * blockIdx.x;
        c[0] = clk_t0; c[1] = __builtin_amdgcn_s_memtime(); c[2] = clk_r0; c[3] = __builtin_amdgcn_s_memrealtime();
    }
}

// The forms, by groups of 16 tokens: eight waves where LDS holds their codes, and the most waves for longer rows. A row of G groups
// takes the first whose waves have room for it. Rows of X in halves of a group where whole ones would leave room for fewer waves: 4096 x 5120
// at 45 / 60 tokens 9.2 / 10.7 us on six and five waves with whole groups, 9.0 / 9.9 on eight with halves.
struct FewForm {
    int waves, groups;  // groups a wave has room for
    bool half;          // rows of X in halves of a group
};
template <int MT>
constexpr int kFewForms = MT <= 3 ? 3 : 2;
template <int MT>
constexpr FewForm few_form(int i) {
    constexpr FewForm forms[5][3] = {{{8, 4, false}, {8, 8, false}, {6, 15, false}}, {{8, 4, false}, {8, 8, true}, {8, 11, true}},
                                     {{7, 5, false}, {8, 8, true}, {}}, {{8, 4, true}, {8, 7, true}, {}}, {{8, 3, true}, {7, 6, true}, {}}};
    return forms[MT <= 4 ? MT - 2 : MT / 2][i];  // 2, 3, 4, 6, 8
}
template <int MT>
constexpr int few_groups() { return few_form<MT>(kFewForms<MT> - 1).waves * few_form<MT>(kFewForms<MT> - 1).groups; }

template <int MT, int I, class Launch>
void few_launch(int G, Launch &&launch) {
    constexpr FewForm f = few_form<MT>(I);
    if constexpr (I + 1 < kFewForms<MT>)
        if (G > f.waves * f.groups) return few_launch<MT, I + 1>(G, launch);
    if constexpr (!f.half) launch(gemm_few_kernel<MT, f.groups, f.waves>, f.waves);
    else launch(gemm_few_half_kernel<MT, f.groups, f.waves>, f.waves);
}

}  // namespace

// The longest row, in groups of 128 k, that the kernel takes for M tokens (0: none)
int lq_gemm_few_groups(long long M) {
    return M <= 16 || M > 128 ? 0 : M <= 32 ? few_groups<2>() : M <= 48 ? few_groups<3>() : M <= 64 ? few_groups<4>() : M <= 96 ? few_groups<6>() : few_groups<8>();
}

// 16 < M <= 128, N % 16 == 0, K % 128 == 0 and K / 128 <= lq_gemm_few_groups(M) are guaranteed by the caller.
int lq_gemm_few_launch(const void *x, const void *codes, const void *scales, const void *zeros, const void *bias, void *y, int M, int N,
                       int K, hipStream_t st, unsigned long long *clk, const char *who) {
    // what the waves' LDS holds (and with it the 32-bit lane offsets of the loads, which span the tokens' rows and 16 rows of codes)
    if (K / LQ_GROUP > lq_gemm_few_groups(M)) return lq_fail(LQ_ERR_BAD_ARG, "%s: K too large", who);
    auto launch = [&](auto kernel, int waves) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(N / 16)), dim3(64 * waves), 0, st, (const unsigned char *)x, (const unsigned char *)codes, M, N, K,
                           (const unsigned short *)scales, (const unsigned short *)zeros, (const unsigned short *)bias, (unsigned short *)y, clk);
    };
    if (M <= 32) few_launch<2, 0>(K / LQ_GROUP, launch);
    else if (M <= 48) few_launch<3, 0>(K / LQ_GROUP, launch);
    else if (M <= 64) few_launch<4, 0>(K / LQ_GROUP, launch);
    else if (M <= 96) few_launch<6, 0>(K / LQ_GROUP, launch);
    else few_launch<8, 0>(K / LQ_GROUP, launch);
    return lq_check_launch(who);
}
