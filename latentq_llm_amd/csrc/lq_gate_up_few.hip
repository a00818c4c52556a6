// h = silu(X Wgate^T) * (X Wup^T) for 17 to 64 tokens and up to 32 columns per compute unit, in one launch.
//
// Bound: vector issue of the conversion (19 instructions per 8 weights), the MFMAs and the loads, one after the other in a wave and beside
// another wave's. The staged kernel (lq_gemm_staged.hip) fills the device with such an output only by cutting K, and the launch that
// adds the slices takes as long as the product; whole, its tiles of 64 columns of both matrices leave units idle, and its waves
// meet at a barrier for every pair of groups. Here a workgroup owns 16 NB columns of both matrices, all tokens and all of K; its eight waves
// each take a contiguous share of the groups of 128 k, on their own loads and waits, and their sums meet in LDS once, in the order
// of k. Every workgroup reads all of X from L2.
//
// us, weights from HBM, staged kernel -> this one:
//     N x K          20 tokens        33               45               60
//     4096 x 2048    11.0 -> 6.4      12.3 -> 7.3      13.0 -> 7.2      10.3 -> 8.4
//     2816 x 1024    6.8 -> 4.3       7.0 -> 4.9       7.1 -> 4.9       7.1 -> 5.5
//     5504 x 2048    10.9 -> 8.6      12.2 -> 9.6      10.5 -> 9.5      (10.5, 11.6)
//     7168 x 3584    14.4 -> 13.3     16.4 -> 15.6     16.9 -> 15.7     (18.3, 20.5)
// With NB = 3 (11008 x 4096 at 17 / 45 / 64 tokens 19.2 / 22.5 / 25 against 19.3 / 21.5 / 21.7) it gains nothing: what a unit converts is
// what it has to convert in either kernel. Also measured there: no loads after the first group 19.0, no conversion 17.8, neither 12.7, codes in
// registers and across lanes by ds_bpermute 22.0, 17 instructions per 8 weights with v_fma_mix_f32 23.0.
#include "lq_common.h"

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef unsigned u32x2_a4_t __attribute__((ext_vector_type(2), aligned(4)));

constexpr int kWaves = 8;
constexpr int kHeldGroups = 7;  // groups of a wave, at most: a lane pair holds eight scales, of which the first may be one too early

// LDS: a wave's rows of X and codes of one group; at the end the sums of all waves
constexpr int gate_up_few_lds(int MT, int NB) {
    const int staged = kWaves * (MT * 4096 + 2 * NB * 1024), sums = kWaves * 2 * NB * MT * 1024;
    return staged > sums ? staged : sums;
}

// MT: groups of 16 tokens. MFMA 16x16x32, weights first: lane l holds token l % 16 of four consecutive columns. With r = l % 16,
// h = l / 16 slice w = 0..3 of a group has the lane's operands at k = 32 h + 8 w .. + 7: word w of 16 bytes of codes of row r, and a
// 16-byte piece of X. A wave has LDS of its own for one group: 16 MT rows of X of 256 bytes, piece c of row i at c ^ (i & 15), and 2 NB
// blocks of 16 rows of codes of 64 bytes, piece c of row i at c ^ ((i >> 2) & 3). They are read into registers and replaced by the
// next group's before the products begin.
template <int MT, int NB>
__global__ __launch_bounds__(64 * kWaves) void gate_up_few_kernel(
    const unsigned char *x, const unsigned char *wg, const unsigned char *wu, int M, int N, int K, const unsigned short *sg,
    const unsigned short *zg, const unsigned short *su, const unsigned short *zu, unsigned short *h_out, unsigned short *g_out,
    unsigned short *u_out) {
    constexpr int B = 2 * NB;  // blocks of 16 columns: the gate's, then the up projection's
    __shared__ __attribute__((aligned(16))) unsigned char lds[gate_up_few_lds(MT, NB)];
    static_assert(sizeof(lds) <= 160 << 10, "LDS");
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, r = lane & 15, h = lane >> 4;
    const int G = K / LQ_GROUP;
    unsigned char *const rows = lds + wave * (MT * 4096 + B * 1024), *const codes = rows + MT * 4096;
    const int share = G / kWaves, more = G % kWaves;
    const int ng = share + (wave < more ? 1 : 0), g0 = wave * share + (wave < more ? wave : more);
    auto column = [&](int b) {  // first column of the block (past the matrix: the last one again, not stored)
        const int c = (blockIdx.x * NB + b % NB) * 16;
        return c < N ? c : N - 16;
    };

    // ---- loads
    // scales on lanes 0..15 and 32..47, zeros on the others: four values each, from an even index of the row on
    const int q0 = (g0 & ~1) < G - 8 ? g0 & ~1 : G - 8;
    u32x2_t q[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        const unsigned short *s = b < NB ? sg : su, *z = b < NB ? zg : zu;
        q[b] = *reinterpret_cast<const u32x2_a4_t *>((h & 1 ? z : s) + (long long)(column(b) + r) * G + q0 + 4 * (h >> 1));
    }
    const int crow = lane >> 2;
    const unsigned c_off = (unsigned)crow * (unsigned)(K / 2) + ((lane & 3) ^ ((crow >> 2) & 3)) * 16;
    auto load_codes = [&](int g) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(codes + b * 1024));
            const unsigned char *src = (b < NB ? wg : wu) + (long long)column(b) * (K / 2) + g * 64;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(c_off), "s"(src) : "memory");
        }
    };
    // load i brings rows 4 i .. 4 i + 3; past the last token: that one's again. Of the rows before the last 16 all are there.
    const unsigned lda = (unsigned)K * 2u;
    unsigned a_last[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 16 * (MT - 1) + 4 * i + h;
        a_last[i] = (unsigned)(row < M ? row : M - 1) * lda + (r ^ (row & 15)) * 16;
    }
    const unsigned a_first = (unsigned)h * lda + (r ^ h) * 16;
    auto load_rows = [&](int g) {
#pragma unroll
        for (int i = 0; i < 4 * MT; ++i) {
            const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(rows + i * 1024));
            const bool last = i >= 4 * (MT - 1);
            const unsigned off = last ? a_last[i & 3] : a_first ^ ((i & 3) * 64);  // (rows are multiples of 256 bytes)
            const unsigned char *src = x + (long long)g * 256 + (last ? 0ll : (long long)(4 * i) * lda);
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
        }
    };

    f32x4_t acc[B][MT];
#pragma unroll
    for (int b = 0; b < B; ++b)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[b][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    load_codes(g0);
    load_rows(g0);
#pragma unroll
    for (int b = 0; b < B; ++b) asm volatile("" : "+v"(q[b]));  // (the compiler would wait for them inside the loop, and so for the loads ahead)
    for (int i = 0; i < ng; ++i) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        u32x4_t c[B];
#pragma unroll
        for (int b = 0; b < B; ++b) c[b] = *reinterpret_cast<const u32x4_t *>(codes + b * 1024 + r * 64 + ((h ^ ((r >> 2) & 3)) << 4));
        u32x4_t xv[4][MT];
#pragma unroll
        for (int w = 0; w < 4; ++w)
#pragma unroll
            for (int j = 0; j < MT; ++j) xv[w][j] = *reinterpret_cast<const u32x4_t *>(rows + (16 * j + r) * 256 + (((4 * h + w) ^ r) << 4));
        // the place of the rows and of the codes is free once these reads have returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (i + 1 < ng) {
            load_codes(g0 + i + 1);
            load_rows(g0 + i + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        const int iq = g0 + i - q0, q_src = (r + 32 * (iq >> 2)) * 4;
#pragma unroll
        for (int b = 0; b < B; ++b) {
            const unsigned two = iq & 2 ? q[b][1] : q[b][0];
            const unsigned s2 = (unsigned)__builtin_amdgcn_ds_bpermute(q_src, (int)two), z2 = (unsigned)__builtin_amdgcn_ds_bpermute(q_src + 64, (int)two);
            const float s = lq_bf16_lo(s2 >> (16 * (iq & 1))), z = lq_bf16_lo(z2 >> (16 * (iq & 1)));
            const float s512 = 512.0f * s, nzs = -(z * s);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                float f[8];
                lq_dequant_word_f32(c[b][w], s512, nzs, f);
                const u32x4_t op = {lq_pack_bf16(f[0], f[1]), lq_pack_bf16(f[2], f[3]), lq_pack_bf16(f[4], f[5]), lq_pack_bf16(f[6], f[7])};
#pragma unroll
                for (int j = 0; j < MT; ++j)
                    acc[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, op), __builtin_bit_cast(bf16x8_t, xv[w][j]),
                                                                       acc[b][j], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- partial sums [block][wave][gate, up][16 tokens][lane]
    f32x4_t *const part = reinterpret_cast<f32x4_t *>(lds);
    __syncthreads();
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            f32x4_t *at = part + ((n * kWaves + wave) * 2 * MT + j) * 64 + lane;
            at[0] = acc[n][j];
            at[MT * 64] = acc[NB + n][j];
        }
    __syncthreads();
    for (int t = threadIdx.x; t < NB * MT * 64; t += 64 * kWaves) {
        const int n = t / (MT * 64), jl = t % (MT * 64), l = jl & 63;
        f32x4_t g = {0.f, 0.f, 0.f, 0.f}, u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const f32x4_t *at = part + (n * kWaves + w) * 2 * MT * 64 + jl;
            const f32x4_t a = at[0], b = at[MT * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) { g[e] += a[e]; u[e] += b[e]; }
        }
        const int m = jl / 64 * 16 + (l & 15), c = (blockIdx.x * NB + n) * 16 + 4 * (l >> 4);
        if (m >= M || c >= N) continue;
        const long long at = (long long)m * N + c;
        float o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = g[e] * __builtin_amdgcn_rcpf(1.0f + __expf(-g[e])) * u[e];
        *reinterpret_cast<u32x2_t *>(h_out + at) = u32x2_t{lq_pack_bf16(o[0], o[1]), lq_pack_bf16(o[2], o[3])};
        if (g_out) {
            *reinterpret_cast<u32x2_t *>(g_out + at) = u32x2_t{lq_pack_bf16(g[0], g[1]), lq_pack_bf16(g[2], g[3])};
            *reinterpret_cast<u32x2_t *>(u_out + at) = u32x2_t{lq_pack_bf16(u[0], u[1]), lq_pack_bf16(u[2], u[3])};
        }
    }
}

}  // namespace

// Whether the kernel takes the sizes: shares of K that its waves can hold the scales of, scales and zeros in pairs, a form for the columns
bool lq_gate_up_few_fits(long long M, long long N, long long K, long long cus) {
    const long long G = K / LQ_GROUP;
    return M > 16 && M <= 64 && G >= 8 && G <= kWaves * kHeldGroups && G % 2 == 0 && N <= (M <= 48 ? 32 : 16) * cus;
}

// lq_gate_up_few_fits, N % 16 == 0 and scales and zeros on 4 bytes are guaranteed by the caller.
int lq_gate_up_few_launch(const void *x, const void *codes_g, const void *scales_g, const void *zeros_g, const void *codes_u,
                          const void *scales_u, const void *zeros_u, void *h, void *g_out, void *u_out, int M, int N, int K, hipStream_t st,
                          const char *who) {
    const int cus = lq_device_cu_count();
    if (!lq_gate_up_few_fits(M, N, K, cus)) return lq_fail(LQ_ERR_BAD_ARG, "%s: no kernel for the size", who);
    auto launch = [&](auto kernel, int nb) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((N / 16 + nb - 1) / nb)), dim3(64 * kWaves), 0, st, (const unsigned char *)x,
                           (const unsigned char *)codes_g, (const unsigned char *)codes_u, M, N, K, (const unsigned short *)scales_g,
                           (const unsigned short *)zeros_g, (const unsigned short *)scales_u, (const unsigned short *)zeros_u,
                           (unsigned short *)h, (unsigned short *)g_out, (unsigned short *)u_out);
    };
    if (N / 16 <= cus) {
        if (M <= 32) launch(gate_up_few_kernel<2, 1>, 1);
        else if (M <= 48) launch(gate_up_few_kernel<3, 1>, 1);
        else launch(gate_up_few_kernel<4, 1>, 1);
    } else {
        if (M <= 32) launch(gate_up_few_kernel<2, 2>, 2);
        else launch(gate_up_few_kernel<3, 2>, 2);
    }
    return lq_check_launch(who);
}
