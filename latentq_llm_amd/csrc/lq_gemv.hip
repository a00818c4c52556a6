// Kernel (2b): A16W4 GEMV for decode-sized M (1..16 tokens) on gfx950.
//
// The weight matrix is streamed from HBM exactly once. A workgroup owns 16 consecutive
// weight rows (output features); its waves split the K dimension by quantisation group
// and combine their partial sums through LDS. Inside a wave the contraction runs on the
// 16x16x32 bf16 MFMA with the (zero-padded) token block as the 16-row operand, because at
// 0.5 byte per weight even one fp32 FMA per weight would outrun the vector ALUs before HBM.
//
// Per group g (128 k) and weight row n the kernel uses
//     sum_k x[m,k] * (q[n,k] - z) * s  =  s * ( P[m,n] - (128 + z) * S[m] )
// with P = sum_k x[m,k] * (128 + q[n,k]) and S = sum_k x[m,k], both accumulated by MFMA:
// the code nibbles become the bf16 numbers 128+q by one AND-OR (bit pattern 0x4300 | q),
// so unpacking costs < 1 VALU operation per weight. The scale is applied in fp32 to the
// per-group sums, i.e. weights are NOT rounded to bf16 first (slightly more accurate than
// the dequantise-then-multiply path).
//
// Memory access. The MFMA wants lane 16*kq + n to hold 8 k of weight row n, which as a load
// pattern would put the 4 lanes of every quad on 4 different rows (64 separate cache-line
// requests per wave instruction). The codes are therefore loaded with lane 4*r + c reading
// 16-byte chunk c of row r (a quad reads 64 contiguous bytes) and moved to the MFMA layout
// with one ds_bpermute per dword. For the same reason the scales and zeros of a batch of 4
// consecutive groups are fetched as one 8-byte load by the 16 lanes kq = 0 only and then
// broadcast, and activation loads are limited to the lanes of live tokens: what a vector load
// costs here is cache-line look-ups per quad, not bytes.
#include "lq_common.h"
#include "lq_gemv_batches.h"

namespace {

// k-slot order produced by the AND-OR unpack of one code word: slots (2i, 2i+1) of dword i
// hold codes (1,5), (0,4), (3,7), (2,6). The activation fragment is permuted to match.
__device__ __forceinline__ void unpack_word_128q(unsigned w, unsigned o[4]) {
    o[0] = (w & 0x000F000Fu) | 0x43004300u;
    o[1] = ((w >> 4) & 0x000F000Fu) | 0x43004300u;
    o[2] = ((w >> 8) & 0x000F000Fu) | 0x43004300u;
    o[3] = ((w >> 12) & 0x000F000Fu) | 0x43004300u;
}
__device__ __forceinline__ void permute_x(const u32x4_t &d, unsigned a[4]) {
    a[0] = __builtin_amdgcn_perm(d[2], d[0], 0x07060302u);  // (x1, x5)
    a[1] = __builtin_amdgcn_perm(d[2], d[0], 0x05040100u);  // (x0, x4)
    a[2] = __builtin_amdgcn_perm(d[3], d[1], 0x07060302u);  // (x3, x7)
    a[3] = __builtin_amdgcn_perm(d[3], d[1], 0x05040100u);  // (x2, x6)
}

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void gbl_void;

constexpr int kXRow = 1024 + 16;  // LDS bytes per staged token row: 4 groups x 256 B, padded against bank conflicts
// MP = number of token rows staged per wave and batch (>= M). NT = 16-row weight tiles per
// workgroup: every workgroup stages the activations of its K range again, so with many tokens two
// tiles per workgroup halve that traffic (and share the activation-sum MFMAs).
// GU (with NT = 2, no QS): gate / up mode. Tile 1 is the same 16 rows of a second matrix (codes2, scales2,
// zeros2) and the output is silu(tile 0) * tile 1 on the fp32 sums: the gate / up pair of a gated MLP in one
// pass over both matrices. There batch b goes into partial sum b % slots, a number that the launcher derives from M and K
// alone, and a wave works through up to SPW partial sums one after the other: the order of the fp32 sums, and so the bits of
// the result, do not depend on how many waves the launcher finds best for the grid.
// (SPW = 2 in at most 128 registers, four waves to a SIMD; more in 168)
// LOADS: how a wave's batches are loaded.
//   0  at the top of the loop over them, the token rows by the compiler's LDS-direct load, after which it waits for
//      all loads before any read of LDS
//   1  the same, the token rows by assembly
//   2  the next batch's codes before this one's MFMAs (24 to 32 registers more)
//   3  no loop: one batch a wave. Its loads come before all that is not needed for them; a loop has a hundred
//      instructions in front of it, a twentieth of a small launch
// The arguments that the first loads need come first: the leading 14 dwords are preloaded into registers (build.py). Weights from
// HBM, 1 token: 4096 x 4096 5.15 -> 4.77 us, 4096 x 11008 8.01 -> 7.76, 2048 x 2048 3.48 -> 3.31.
template <int WAVES, int MP, int NT, bool QS, bool GU = false, int SPW = 1, int LOADS = 0>
__global__ __launch_bounds__(64 * WAVES, LOADS >= 2 ? 1 : SPW == 2 ? 4 : SPW > 2 ? 3 : 1) void gemv_kernel(
    const unsigned short *__restrict__ x, const unsigned char *__restrict__ codes, int M, int N, int K, int slots,
    const unsigned short *__restrict__ scales, const unsigned short *__restrict__ zeros, const unsigned short *__restrict__ bias,
    unsigned short *__restrict__ y, const unsigned char *__restrict__ codes2, const unsigned short *__restrict__ scales2,
    const unsigned short *__restrict__ zeros2) {
    constexpr bool PRE = LOADS == 2, ONE = LOADS == 3;
    static_assert(!GU || (NT == 2 && !QS), "gate / up mode: two tiles, scales and zeros straight from memory");
    constexpr int RT = GU ? 1 : NT;  // 16-row tiles of output rows per workgroup
    static_assert(LOADS < 2 || SPW == 1, "one partial sum a wave");
    static_assert(GU || SPW == 1, "several partial sums per wave: gate / up mode only");
    constexpr int kWaveLds = MP * kXRow > SPW * NT * 1024 ? MP * kXRow : SPW * NT * 1024;
    __shared__ __attribute__((aligned(16))) unsigned char xs_all[WAVES][kWaveLds];
    const auto xs = [&](int w, int m) { return &xs_all[w][m * kXRow]; };
    // partial sums [slot of the wave][tile][4][lane] take the place of the token rows the wave staged (its reads of them
    // have returned); slot s is slot s / WAVES of wave s % WAVES
    auto red = [&](int s, int j, int r) -> float & {
        return reinterpret_cast<float *>(&xs_all[s % WAVES][0])[((s / WAVES * NT + j) * 4 + r) * 64 + (threadIdx.x & 63)];
    };
    extern __shared__ __attribute__((aligned(16))) unsigned char sq[];  // QS: scales then zeros of the workgroup's rows
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // scalar: uniform control flow
    const int n = lane & 15, kq = lane >> 4;
    const int row = blockIdx.x * (16 * RT) + n;  // weight row of this lane's B fragment in tile 0 (tile j: + 16 j)
    const int G = K / LQ_GROUP;

    // load layout of the codes: lane 4*r + c -> row r of this block, 16-byte chunk c of the group
    const long long wrow_off = (long long)(blockIdx.x * (16 * RT) + (lane >> 2)) * (K / 2) + (lane & 3) * 16;
    const unsigned char *wrow = codes + wrow_off;
    const unsigned char *wrow2 = GU ? codes2 + wrow_off : nullptr;  // gate / up mode: tile 1 is the second matrix
    const long long tile_stride = 16ll * (K / 2);  // bytes between the same row of consecutive tiles
    const int bperm_src = (4 * n + kq) * 4;  // ds_bpermute: take from lane 4*n + kq
    const int bcast_src = n * 4;             // ds_bpermute: take from lane n (kq = 0)
    const unsigned short *srow = scales + (long long)row * G;
    const unsigned short *zrow = zeros + (long long)row * G;
    // As an A-fragment lane, `n` is the token index; lanes of tokens >= M re-read the last staged
    // row: they only feed accumulator rows m >= M, which are never stored.
    const unsigned char *xfrag = xs(wave, n < M ? n : M - 1) + kq * 64;

    const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
    f32x4_t acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // QS: the scales and zeros of the workgroup's 16*NT rows are one contiguous block each; the waves
    // fetch them together with 16-byte loads (issued first, so that they return first) and every wave
    // then takes its groups from LDS
    constexpr int kQPieces = 2;  // 16-byte pieces per thread: up to 64*WAVES*2*16 bytes of scales + zeros
    const int q_bytes = 16 * NT * G * 2;
    // LDS row pitch of the staged block: rows whose length is a multiple of 16 bytes get 16 bytes of
    // padding (a 64-byte pitch would put the 16 rows a group is read from on 4 bank groups); other
    // lengths keep the block as it is (its 16-byte pieces straddle rows)
    const int q_row = G * 2, q_pitch = (q_row % 16 == 0) ? q_row + 16 : q_row;
    const int q_lds = 16 * NT * q_pitch;  // bytes per array in LDS
    u32x4_t qstage[kQPieces];
    if constexpr (QS) {
        const unsigned char *sb = (const unsigned char *)(scales + (long long)blockIdx.x * (16 * NT) * G);
        const unsigned char *zb = (const unsigned char *)(zeros + (long long)blockIdx.x * (16 * NT) * G);
#pragma unroll
        for (int i = 0; i < kQPieces; ++i) {
            const int pc = (int)threadIdx.x + i * 64 * WAVES;
            const int o = pc * 16;
            qstage[i] = u32x4_t{0u, 0u, 0u, 0u};
            if (o < 2 * q_bytes) qstage[i] = *reinterpret_cast<const u32x4_t *>(o < q_bytes ? sb + o : zb + (o - q_bytes));
        }
    }
    bool first = true;
    // every wave runs this exactly once: in its first batch, after that batch's loads are issued, or
    // after the loop when it has no batch at all (the barrier inside needs all waves)
    auto publish_q = [&]() {
#pragma unroll
        for (int i = 0; i < kQPieces; ++i) {
            const int o = ((int)threadIdx.x + i * 64 * WAVES) * 16;
            if (o < 2 * q_bytes) {
                const int oa = o < q_bytes ? o : o - q_bytes;
                const int dst = q_pitch == q_row ? oa : (oa / q_row) * q_pitch + oa % q_row;
                *reinterpret_cast<u32x4_t *>(sq + (o < q_bytes ? 0 : q_lds) + dst) = qstage[i];
            }
        }
        __syncthreads();
    };
    const int n_slots = GU ? slots : WAVES;
    f32x4_t done[SPW][NT];  // SPW > 1: the wave's complete partial sums
#pragma unroll
    for (int k = 0; k < SPW; ++k)
#pragma unroll
        for (int j = 0; j < NT; ++j) done[k][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto keep = [&](int i) {  // partial sum i is complete
#pragma unroll
        for (int k = 0; k < SPW; ++k)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) done[k][j][r] = i == k ? acc[j][r] : done[k][j][r];
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    // ---- loads of the batch that begins with group g0
    // activations: one LDS-direct load per token row (1 KB = this batch's 512 k), coalesced. In a tail batch the lanes past the
    // end of the row re-read its first bytes (dead groups). LOADS > 0: written as assembly, with which the compiler does not
    // wait for the rows (or the next batch's codes) before each of its own reads of LDS.
    auto load_x = [&](int g0) {
        const long long xoff = (long long)g0 * (LQ_GROUP * 2) + lane * 16;
        const long long lim = (long long)K * 2;
        const long long off = xoff < lim ? xoff : 0;
#pragma unroll
        for (int m = 0; m < MP; ++m)
            if (m < M) {
                const unsigned char *src = (const unsigned char *)x + (long long)m * lim;
                if constexpr (LOADS > 0) {
                    const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)xs(wave, m));
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"((unsigned)off), "s"(src) : "memory");
                } else {
                    __builtin_amdgcn_global_load_lds((gbl_void *)(src + off), (lds_void *)xs(wave, m), 16, 0, 0);
                }
            }
    };
    // codes, and the scales and zeros of a whole batch (loaded by the 16 lanes kq = 0)
    u32x4_t wn[NT][kUnroll];
    u32x2_t sn[NT], zn[NT];
    auto scale_row = [&](int j) { return GU ? (j == 0 ? srow : scales2 + (long long)row * G) : srow + (long long)j * 16 * G; };
    auto zero_row = [&](int j) { return GU ? (j == 0 ? zrow : zeros2 + (long long)row * G) : zrow + (long long)j * 16 * G; };
    auto load_scales = [&](int g0, int j) {
        sn[j] = zn[j] = u32x2_t{0u, 0u};
        if (kq == 0) {
            sn[j] = *reinterpret_cast<const u32x2_t *>(scale_row(j) + g0);
            zn[j] = *reinterpret_cast<const u32x2_t *>(zero_row(j) + g0);
        }
    };
    auto load_codes = [&](int g0) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const int g = g0 + u < G ? g0 + u : G - 1;
                const unsigned char *wt = (GU && j == 1) ? wrow2 : wrow + j * tile_stride;
                wn[j][u] = *reinterpret_cast<const u32x4_t *>(wt + g * 64);
            }
        if constexpr ((PRE || ONE) && !QS)
            if (g0 + kUnroll <= G) {
#pragma unroll
                for (int j = 0; j < NT; ++j) load_scales(g0, j);
            }
    };
    // the batch at group g0, whose loads have been issued; `then` issues what is to travel under its MFMAs and waits for the
    // staged rows
    auto multiply = [&](int g0, auto then) {
        const bool full = g0 + kUnroll <= G;  // a short tail batch re-reads the last group with zero scale
        u32x4_t wv[NT][kUnroll];
        float sc[NT][kUnroll], zz[NT][kUnroll];
        if constexpr (QS) {
            if (first) {
                publish_q();
                first = false;
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const unsigned short *ls = reinterpret_cast<const unsigned short *>(sq + (j * 16 + n) * q_pitch);
                const unsigned short *lz = reinterpret_cast<const unsigned short *>(sq + q_lds + (j * 16 + n) * q_pitch);
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    const bool live = g0 + u < G;
                    const int g = live ? g0 + u : G - 1;
                    sc[j][u] = live ? lq_bf16_bits_to_f32(ls[g]) : 0.0f;
                    zz[j][u] = 128.0f + lq_bf16_bits_to_f32(lz[g]);
                }
            }
        } else if (full) {
            if constexpr (LOADS == 1) {
#pragma unroll
                for (int j = 0; j < NT; ++j) load_scales(g0, j);
            }
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                if constexpr (LOADS == 0) load_scales(g0, j);
                const unsigned s01 = (unsigned)__builtin_amdgcn_ds_bpermute(bcast_src, (int)sn[j][0]);
                const unsigned s23 = (unsigned)__builtin_amdgcn_ds_bpermute(bcast_src, (int)sn[j][1]);
                const unsigned z01 = (unsigned)__builtin_amdgcn_ds_bpermute(bcast_src, (int)zn[j][0]);
                const unsigned z23 = (unsigned)__builtin_amdgcn_ds_bpermute(bcast_src, (int)zn[j][1]);
                sc[j][0] = lq_bf16_lo(s01); sc[j][1] = lq_bf16_hi(s01); sc[j][2] = lq_bf16_lo(s23); sc[j][3] = lq_bf16_hi(s23);
                zz[j][0] = 128.0f + lq_bf16_lo(z01); zz[j][1] = 128.0f + lq_bf16_hi(z01);
                zz[j][2] = 128.0f + lq_bf16_lo(z23); zz[j][3] = 128.0f + lq_bf16_hi(z23);
            }
        } else {
#pragma unroll
            for (int j = 0; j < NT; ++j) {
#pragma unroll
                for (int u = 0; u < kUnroll; ++u) {
                    const bool live = g0 + u < G;
                    const int g = live ? g0 + u : G - 1;
                    sc[j][u] = live ? lq_bf16_bits_to_f32(scale_row(j)[g]) : 0.0f;
                    zz[j][u] = 128.0f + lq_bf16_bits_to_f32(zero_row(j)[g]);
                }
            }
        }
        // ---- codes to the MFMA lane layout
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < kUnroll; ++u)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    wv[j][u][t] = (unsigned)__builtin_amdgcn_ds_bpermute(bperm_src, (int)wn[j][u][t]);
        then();
        // ---- MFMAs
        // One group at a time: a single pair of MFMA accumulators (plus one per extra tile) is live; the unpacking between
        // two MFMAs on the same accumulator covers their latency.
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            f32x4_t P[NT], S = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NT; ++j) P[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                unsigned a[4];
                const u32x4_t xv = *reinterpret_cast<const u32x4_t *>(xfrag + u * 256 + t * 16);
                permute_x(xv, a);
                const u32x4_t av = {a[0], a[1], a[2], a[3]};
                S = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av),
                                                            __builtin_bit_cast(bf16x8_t, ones), S, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    unsigned b[4];
                    unpack_word_128q(wv[j][u][t], b);
                    const u32x4_t bv = {b[0], b[1], b[2], b[3]};
                    P[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av),
                                                                   __builtin_bit_cast(bf16x8_t, bv), P[j], 0, 0, 0);
                }
            }
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[j][r] = fmaf(sc[j][u], fmaf(-zz[j][u], S[r], P[j][r]), acc[j][r]);
            __builtin_amdgcn_sched_barrier(0);  // keeps the next group's unpacking from being hoisted (registers)
        }
        // the next batch overwrites the staged rows: all fragment reads above must have returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };
    if constexpr (ONE) {
        const int g0 = wave * kUnroll;
        if (g0 < G) {
            load_x(g0);
            load_codes(g0);
            __builtin_amdgcn_sched_barrier(0);  // the loads before all that is not needed for them
            multiply(g0, []() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); });
        }
    } else if constexpr (PRE) {
        gemv_batches_ahead(wave, n_slots, G, load_x, load_codes, multiply, []() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); });
    } else {
        for (int i = 0; i < SPW; ++i) {
            const int s = wave + i * WAVES;
            if (SPW > 1 && s >= n_slots) break;
            for (int g0 = s * kUnroll; g0 < G; g0 += n_slots * kUnroll) {
                load_x(g0);
                load_codes(g0);
                multiply(g0, []() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); });
            }
            if constexpr (SPW > 1) keep(i);
        }
    }

    if constexpr (QS) {
        if (first) publish_q();
    }
#pragma unroll
    for (int k = 0; k < SPW; ++k)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) red(wave + k * WAVES, j, r) = SPW > 1 ? done[k][j][r] : acc[j][r];
    __syncthreads();
    if constexpr (GU) {
        if (wave == 0) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float g = 0.f, u = 0.f;
#pragma unroll
                for (int s = 0; s < SPW * WAVES; ++s) {  // (those without a batch are zero)
                    g += red(s, 0, r);
                    u += red(s, NT - 1, r);
                }
                const int m = 4 * kq + r;
                if (m < M) y[(long long)m * N + row] = lq_f32_to_bf16_bits(g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u);
            }
        }
    } else if (wave < NT) {
        // wave j finishes tile j; lane holds D[m = 4*kq + r][n]
        const int orow = row + 16 * wave;
        const float b = bias ? lq_bf16_bits_to_f32(bias[orow]) : 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) v += red(w, wave, r);
            const int m = 4 * kq + r;
            if (m < M) y[(long long)m * N + orow] = lq_f32_to_bf16_bits(v + b);
        }
    }
}

}  // namespace

namespace {

struct GemvArgs {
    const void *x, *codes, *scales, *zeros, *bias;
    void *y;
    int M, N, K;
    hipStream_t st;
};

struct GemvGuArgs {
    const void *x, *codes, *scales, *zeros, *codes2, *scales2, *zeros2;
    void *y;
    int M, N, K;
    int slots;
    hipStream_t st;
};

template <int W, int MP, int SPW, int LOADS>
bool launch_gu_loads(const GemvGuArgs &a) {
    hipLaunchKernelGGL((gemv_kernel<W, MP, 2, false, true, SPW, LOADS>), dim3(a.N / 16), dim3(64 * W), 0, a.st, (const unsigned short *)a.x,
                       (const unsigned char *)a.codes, a.M, a.N, a.K, a.slots, (const unsigned short *)a.scales, (const unsigned short *)a.zeros,
                       (const unsigned short *)nullptr, (unsigned short *)a.y, (const unsigned char *)a.codes2,
                       (const unsigned short *)a.scales2, (const unsigned short *)a.zeros2);
    return true;
}

// How the batches are loaded (LOADS): with one workgroup to a unit registers are free for the next batch's codes; with two they
// are not, and with three and more than 4 rows the rows' wait for all loads does no harm (8 tokens, 11008 x 4096: 15.9 us
// against 17.1 by assembly). us, all by the compiler's loads (what every size took before) -> this rule:
//   4096 x 2048 (c = 1)  2 tokens 5.92 -> 5.47, 12: 6.62 -> 5.97;  4096 x 1792, 8: 6.19 -> 5.46;  3072 x 1024, 16: 5.33 -> 5.01
//   6144 x 3072 (c = 2)  8: 10.6 -> 9.94, 12: 12.8 -> 11.4, 16: 12.6 -> 11.9;  8192 x 4096, 12: 15.4 -> 13.3, 16: 15.6 -> 14.2
//   8192 x 2560, 1: 9.2 -> 8.1;  11008 x 4096 (c = 3), 1: 14.2 -> 13.1, 4: 15.1 -> 14.5;  20480 x 8192, 1: 50.1 -> 46.3
// Only the forms that gu_waves can ask for are there: with c = 1 every partial sum has a wave of its own, as with c = 2 and 8 rows;
// with more rows or workgroups the waves are as few as the bounds below say. False for any other form.
template <int W, int MP, int SPW>
bool launch_gu_spw(const GemvGuArgs &a) {
    if constexpr (MP == 4) {
        return launch_gu_loads<W, MP, SPW, 1>(a);
    } else {
        const int c = (a.N / 16 + lq_device_cu_count() - 1) / lq_device_cu_count();
        if constexpr (SPW == 1)
            if (c == 1) return launch_gu_loads<W, MP, SPW, 2>(a);
        if constexpr (MP == 8 ? SPW == 1 : W <= 4 && SPW <= 2 && W > SPW)
            if (c == 2) return launch_gu_loads<W, MP, SPW, 1>(a);
        if constexpr (W <= (MP == 16 ? 3 : MP == 12 ? 4 : 5))
            if (c > 2) return launch_gu_loads<W, MP, SPW, 0>(a);
        return false;
    }
}

// Partial sums of a gate / up pass, at most: the waves of the workgroups that stage 4 or 16 rows with one batch each
constexpr int gu_max_slots(int MP) { return MP == 4 ? 16 : 8; }

template <int W, int MP>
bool launch_gu(const GemvGuArgs &a) {
    constexpr int kMost = (gu_max_slots(MP) + W - 1) / W;
    const int batches = (a.K / LQ_GROUP + kUnroll - 1) / kUnroll, used = batches < a.slots ? batches : a.slots;
    const int spw = (used + W - 1) / W;
    if (spw <= 1) return launch_gu_spw<W, MP, 1>(a);
    if constexpr (kMost >= 2)
        if (spw == 2) return launch_gu_spw<W, MP, 2>(a);
    if constexpr (MP >= 12 && kMost > 2) return launch_gu_spw<W, MP, kMost>(a);
    return false;
}

// Waves per workgroup of the gate / up pass, MP staged rows. A grid of c workgroups per CU should be resident at once: the
// staged rows (1040 MP bytes a wave) of c of them have to fit the CU's 160 KB and their waves its registers (16 of this
// kernel). Within that the fewest rounds of batches, and the fewest waves for that number of rounds. us, 8 waves (what
// every size took before) -> this rule, both matrices:
//   11008 x 4096 (c = 3)  1 token 16.7 -> 15.3 (4 waves), 8: 24.2 -> 16.4 (4), 12: 25.0 -> 17.5 (4), 16: 25.3 -> 20.3 (3)
//   8192 x 2560 (c = 2)   8: 14.9 -> 10.7 (5), 12: 15.0 -> 12.7 (3), 16: 15.3 -> 13.1 (3)
//   6144 x 3072 (c = 2)   8: 14.4 -> 11.2 (6), 12: 14.7 -> 12.7 (3), 16: 15.1 -> 13.2 (3)
// (12 rows and more on 5 or 6 waves are slower although two such workgroups fit: 6144 x 3072 at 12 tokens 11.7 on 6.)
int gu_waves(int MP, int N, int batches, int slots, int cus) {
    const int c = (N / 16 + cus - 1) / cus;
    int most = (160 << 10) / c / (MP * kXRow);
    if (c > 1 && most > 16 / c) most = 16 / c;
    if (c > 1 && MP >= 12 && most > 4) most = 4;
    if (most > (MP == 4 ? 16 : 8)) most = MP == 4 ? 16 : 8;
    if (most < 2) most = 2;
    int w = 2;
    if (batches > slots) {  // a partial sum has several batches, all of one wave: the fewest rounds of wave 0, which has the most
        int best_rounds = 1 << 30;
        for (int c : {2, 3, 4, 5, 6, 8, 16}) {
            int rounds = 0;
            for (int s = 0; s < slots; s += c) rounds += (batches - s + slots - 1) / slots;
            if (c <= most && rounds < best_rounds) { w = c; best_rounds = rounds; }
        }
    } else {
        const int rounds = (batches + most - 1) / most;
        w = (batches + rounds - 1) / rounds;
    }
    // More than two partial sums a wave cost few tokens more than workgroups that wait for a place: 20480 x 8192 at 1 token 61
    // us on 3 waves, 48 on 8; 20480 x 4096 32.3 on 3, 25.4 on 4.
    const int used = batches < slots ? batches : slots;
    if (MP <= 8 && w < (used + 1) / 2) w = (used + 1) / 2;
    return w < 2 ? 2 : w <= 6 ? w : w <= 8 ? (most >= 8 || MP <= 8 ? 8 : 6) : 16;
}

template <int MP>
bool launch_gu_waves(int w, const GemvGuArgs &a) {
    switch (w) {
        case 2: return launch_gu<2, MP>(a);
        case 3: return launch_gu<3, MP>(a);
        case 4: return launch_gu<4, MP>(a);
        case 5: return launch_gu<5, MP>(a);
        case 6: return launch_gu<6, MP>(a);
        case 8: return launch_gu<8, MP>(a);
        default: if constexpr (MP == 4) return launch_gu<16, MP>(a); else return launch_gu<8, MP>(a);
    }
}

// ONE, LOOP: whether pick_waves takes W for so many batches (one each at most) and for more of them; only what can be launched is there.
template <int W, int MP, int NT, bool ONE, bool LOOP>
void launch_one(const GemvArgs &a) {
    // Scales and zeros through LDS: pays with many staged tokens when a wave uses them for more than one
    // batch or for two row tiles (measured: 13.5 -> 12.5 us on 11008 x 4096 at 16 tokens; with one batch
    // and one tile per wave the extra barrier costs more than the loads it saves). Both blocks must be
    // 16-byte aligned and fit two 16-byte pieces per thread.
    const size_t q_bytes = (size_t)16 * NT * (a.K / LQ_GROUP) * 2;
    const int batches = (a.K / LQ_GROUP + kUnroll - 1) / kUnroll;
    const bool qs = MP == 16 && (NT == 2 || batches > W) && lq_aligned(a.scales, 16) && lq_aligned(a.zeros, 16) &&
                    2 * q_bytes <= (size_t)64 * W * 2 * 16;
    auto launch = [&](auto kernel, size_t lds) {
        hipLaunchKernelGGL(kernel, dim3(a.N / (16 * NT)), dim3(64 * W), lds, a.st, (const unsigned short *)a.x, (const unsigned char *)a.codes,
                           a.M, a.N, a.K, W, (const unsigned short *)a.scales, (const unsigned short *)a.zeros, (const unsigned short *)a.bias,
                           (unsigned short *)a.y, (const unsigned char *)nullptr, (const unsigned short *)nullptr, (const unsigned short *)nullptr);
    };
    // How the batches are loaded (LOADS). us, all by the compiler's loads in a loop (what every size took before) -> this rule:
    //   one batch a wave        12 tokens, 4096 x 4096 5.95 -> 5.72; 3 tokens, 1280 x 3584 3.94 -> 3.83; 1 token, 32000 x 4096 17.7 -> 17.1
    //   several, one workgroup  12 tokens, 4096 x 11008 12.7 -> 12.0; 16: 3328 x 9088 11.6 -> 10.5, 2560 x 7680 9.5 -> 8.5,
    //   to a unit               8192 x 4096 10.9 -> 8.8; 10: 2304 x 6144 6.65 -> 6.15; 8: 2048 x 5504 5.9 -> 5.7
    //   16 waves (4096 x 11008, up to 8 tokens) have no registers for a second batch, 7.7 -> 8.4 with it at 1 token
    //   two row tiles           12 tokens, 11008 x 4096 12.3 -> 11.5
    const size_t qs_lds = 2 * q_bytes + 2 * 16 * NT * 16;
    if constexpr (ONE) {
        if (batches <= W) {
            if constexpr (NT == 2)
                if (qs) return launch(gemv_kernel<W, MP, NT, true, false, 1, 3>, qs_lds);
            return launch(gemv_kernel<W, MP, NT, false, false, 1, 3>, 0);
        }
    }
    if constexpr (LOOP) {
        if constexpr (W <= 8) {
            if (a.N / (16 * NT) <= lq_device_cu_count()) {
                if constexpr (MP == 16)
                    if (qs) return launch(gemv_kernel<W, MP, NT, true, false, 1, 2>, qs_lds);
                return launch(gemv_kernel<W, MP, NT, false, false, 1, 2>, 0);
            }
        }
        if constexpr (MP == 16)
            if (qs) return launch(gemv_kernel<W, MP, NT, true, false, 1, NT == 2 ? 1 : 0>, qs_lds);
        launch(gemv_kernel<W, MP, NT, false, false, 1, NT == 2 ? 1 : 0>, 0);
    }
}

// Waves per workgroup: as many as there are batches, up to the cap, in powers of two. More waves
// mean more of the matrix in flight at once, which matters more than an even split of the batches
// (K = 11008 = 22 batches: 16 waves, 6 of them with two batches, beat 11 waves x 2).
int pick_waves(int batches, int max_waves) {
    int w = 2;
    while (w < batches && w < max_waves) w *= 2;
    return w;
}

// As many waves as pick_waves finds for a cap of MAXW (8 rows: of 8 up to 16 batches, of 16 beyond)
template <int MP, int NT, int MAXW>
void launch_waves(const GemvArgs &a, int batches) {
    const int w = pick_waves(batches, MP == 8 && batches <= 16 ? 8 : MAXW);
    if (w == 2) return launch_one<2, MP, NT, true, false>(a);
    if (w == 4) return launch_one<4, MP, NT, true, MAXW == 4>(a);
    if constexpr (MAXW >= 8)
        if (w == 8) return launch_one<8, MP, NT, true, MAXW == 8 || MP == 8>(a);
    if constexpr (MAXW == 16) launch_one<16, MP, NT, MP != 8, true>(a);
}

}  // namespace

int lq_gemv_a16w4_launch(const void *x, const void *codes, const void *scales, const void *zeros, const void *bias,
                         void *y, int M, int N, int K, hipStream_t st) {
    // N % 16 == 0, K % 128 == 0 and 1 <= M <= 16 are guaranteed by the caller.
    const GemvArgs a = {x, codes, scales, zeros, bias, y, M, N, K, st};
    const int batches = (K / LQ_GROUP + 3) / 4;  // one batch of 4 groups per wave when possible: all of a
                                                 // wave's loads are then in flight at once
    if (M <= 4) {
        launch_waves<4, 1, 16>(a, batches);
    } else if (M <= 8) {
        // 8 staged token rows (8.1 KB of LDS per wave): 8 waves with one 16-row tile, 16 when K has more than 16
        // batches (measured on 11008 x 4096 / 4096 x 11008 / 8192^2 at 8 tokens: 11.1 / 10.9 / 14.9 us against
        // 12.1 / 11.8 / 18.5 with 16 staged rows and the two-tile workgroups below)
        launch_waves<8, 1, 16>(a, batches);
    } else if (N % 32 == 0 && N >= 32 * 256) {
        // many tokens and enough rows for one 32-row workgroup per CU: half the activation traffic;
        // 4 waves = 65 KB of staged activations: two workgroups per CU, all of them resident at once
        launch_waves<16, 2, 4>(a, batches);
    } else if (M <= 12 && batches > 8) {
        // (11.4 -> 10.8 us on 4096 x 11008 at 12 tokens, 8.6 -> 7.8 on 2560 x 8192: the loads of four dead rows)
        launch_one<8, 12, 1, false, true>(a);
    } else {
        // 16 staged token rows cost a wave 16.25 KB of LDS, which caps the workgroup at 8 waves
        launch_waves<16, 1, 8>(a, batches);
    }
    return lq_check_launch("lq_a16w4_fwd(gemv)");
}

// silu(x Wgate^T) * (x Wup^T) for 1 <= M <= 16: both matrices in one pass. N % 16 == 0 and K % 128 == 0 are
// guaranteed by the caller.
int lq_gemv_a16w4_gate_up_launch(const void *x, const void *codes_g, const void *scales_g, const void *zeros_g,
                                 const void *codes_u, const void *scales_u, const void *zeros_u, void *h, int M, int N, int K,
                                 hipStream_t st) {
    const int batches = (K / LQ_GROUP + 3) / 4, cus = lq_device_cu_count();
    const int mp = (M + 3) / 4 * 4;
    const int slots = pick_waves(batches, gu_max_slots(mp));
    const GemvGuArgs a = {x, codes_g, scales_g, zeros_g, codes_u, scales_u, zeros_u, h, M, N, K, slots, st};
    const int w = gu_waves(mp, N, batches, slots, cus);
    const bool there = mp == 4 ? launch_gu_waves<4>(w, a) : mp == 8 ? launch_gu_waves<8>(w, a)
                       : mp == 12 ? launch_gu_waves<12>(w, a) : launch_gu_waves<16>(w, a);
    if (!there) return lq_fail(LQ_ERR_BAD_ARG, "lq_a16w4_gate_up_silu(gemv): no kernel of %d waves and %d rows", w, mp);
    return lq_check_launch("lq_a16w4_gate_up_silu(gemv)");
}
