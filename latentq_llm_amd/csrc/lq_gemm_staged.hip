// Forward GEMM of the A16W4 layers with both operands staged in LDS, for grids of few workgroups:
//   Y[M,N] = X[M,K] . deq(W)[N,K]^T (+ bias), or the fp32 partial products of slices of K
//
// 17 to some 500 tokens: a compute unit gets one or two workgroups, so nothing hides a load behind another
// workgroup's work and the time is that of the serial chain through one workgroup's slice of K. What the kernel
// does about it:
//   * a stage is a whole group of 128 k (activations, codes, scales and zeros, all by LDS-direct loads), three stages
//     deep: two groups of loads are in flight while one is multiplied, with one barrier per 128 k;
//   * codes stay packed in LDS (64 bytes per column and group) and each of the four waves converts the 32 columns
//     it multiplies, in registers: no second trip through LDS and no waves that only convert;
//   * a plain product of up to 64 tokens (128 without a workspace) does not round its weights to bf16, since the GEMV, which
//     ran many of these sizes before, does not either: the operand is the integer q - rint(z), exact in bf16, and the scale is
//     applied in fp32 to the sum of a group. Zeros that are no integers of at most 240 add a second product with the
//     remainder (`rest` below). Against the weights as they are a result is 1.66e-3 off, its own rounding, instead of 2.22e-3;
//     it takes 2 to 6 % longer (32 / 64 tokens, 11008 x 4096: 17.1 / 19.7 -> 17.7 / 20.7 us, 4096 x 11008: 17.0 / 19.4 -> 17.4 /
//     20.1; with 128 rows it would be 20 %);
//   * the row tile is 32, 64 or 128 tokens, so that few tokens are not mostly padding; the planner below picks it
//     together with the number of slices of K.
// Bound: LDS reads for 128 rows (one 16-byte fragment read per MFMA), the latency of the chain for 32 and 64.
// Measured, weights from HBM, against the 128 x 128 kernel with separate weight waves that stood here before (and
// 16-token GEMV launches up to 32 tokens), us:
//     N x K           45 tokens       64            128           384
//     4096 x 4096     15.4 -> 11.2    16.0 -> 11.8  20.8 -> 15.4  27.9 -> 23.6
//     11008 x 4096    25.7 -> 17.8    26.4 -> 18.4  28.5 -> 23.4  (weights-direct kernel)
//     4096 x 11008    21.8 -> 15.9    22.0 -> 16.6  25.3 -> 22.6  60.2 -> 51.2
//     2048 x 2048     10.4 -> 7.8     10.8 -> 8.3   12.9 -> 9.6   17.7 -> 11.9
#include "lq_common.h"

#include <type_traits>

namespace {

struct StagedParams {
    const unsigned char *x;  // bf16 [M, K]
    const unsigned char *w;  // packed codes
    const unsigned short *scales, *zeros, *bias;
    // a second matrix of the same shape on the same activations (blockIdx.z = 1), or null: both give partial products
    const unsigned char *w2;
    const unsigned short *scales2, *zeros2;
    unsigned short *y;       // bf16 [M, N]
    float *partial;          // partial products: fp32 [matrices][splits][M][N], or null
    int M, N, K;
    int tiles_m, tiles_n;
    int groups_per_split;    // groups of 128 k per slice (blockIdx.y)
    unsigned long long *clk; // measurement aid, see lq_calib_gemm_clocks; null in normal use
};

typedef __attribute__((address_space(3))) void lds_void;

template <int I>
using ic = std::integral_constant<int, I>;

constexpr int kCols = 128;
constexpr int kCodeBytes = kCols * 64, kScaleBytes = kCols * 4 * 2;
// LDS stages of one group each; a fourth changes nothing, with two the 128-row tile takes 15 % longer
constexpr int D = 3;

// LDS layout of a stage (every 16-byte piece swizzled so that the fragment reads, one piece of 32 consecutive rows,
// spread over all banks):
//   activations  32 FM rows of 256 bytes, chunk c of row i at c ^ (i & 15)
//   codes        128 rows of 64 bytes,   chunk c of row i at c ^ ((i >> 2) & 3)
//   scales, zeros  one dword per column each, the bf16 value in its lower half
// FM: 32-row fragments of the row tile (32 FM rows)
// EXACT: weights as they are (see the top of the file), else rounded to bf16 like those of the kernels for more tokens
// Arguments: those of the first loads first (the leading 14 dwords are preloaded into registers, build.py)
// (launch bounds: with two waves per SIMD asked for, the products of FM < 4 go to vector registers, which the scaling can read)
template <int FM, bool EXACT>
__global__ __launch_bounds__(256, FM < 4 ? 2 : 1) void gemm_staged_kernel(
    const unsigned char *x_, const unsigned char *w_, int M, int N, int K, int tiles_m, int tiles_n, int groups_per_split,
    const unsigned short *scales, const unsigned short *zeros, float *partial, const unsigned short *bias_, unsigned short *y,
    const unsigned char *w2, const unsigned short *scales2, const unsigned short *zeros2, unsigned long long *clk) {
    const StagedParams p = {x_, w_, scales, zeros, bias_, w2, scales2, zeros2, y, partial, M, N, K, tiles_m, tiles_n, groups_per_split, clk};
    constexpr int BM = 32 * FM;
    constexpr int A_BYTES = BM * 256;
    constexpr int STAGE = A_BYTES + kCodeBytes + kScaleBytes;
    constexpr int LA = A_BYTES / 16 / 256;        // loads per thread and stage: activations
    constexpr int LOADS = LA + 2 + 1;             // + codes + one scale or zero
    __shared__ __attribute__((aligned(16))) unsigned char lds[D * STAGE];

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    unsigned long long clk_t0 = 0, clk_r0 = 0;
    if (p.clk) {
        clk_t0 = __builtin_amdgcn_s_memtime();
        clk_r0 = __builtin_amdgcn_s_memrealtime();
    }
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 31, h = lane >> 5;

    const int nwg = p.tiles_m * p.tiles_n;
    int id = blockIdx.x;
    {
        const int per = nwg / 8;
        if (id < per * 8) id = (id % 8) * per + id / 8;
    }
    // row tiles of a column tile follow each other: the weights are read from HBM once
    const int tile_m = id % p.tiles_m, tile_n = id / p.tiles_m;
    const int m0 = tile_m * BM, c0 = tile_n * kCols;
    const int G = p.K / LQ_GROUP;
    const int g0 = p.partial ? (int)blockIdx.y * p.groups_per_split : 0;
    const int g1 = p.partial && g0 + p.groups_per_split < G ? g0 + p.groups_per_split : G;
    const int ng = g1 - g0;

    // ---- loads
    unsigned a_off[LA], c_off[2], q_off;
    const unsigned lda = (unsigned)p.K * 2u, ldw = (unsigned)p.K / 2u;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int s = i * 256 + tid, row = s >> 4, chunk = (s & 15) ^ (row & 15);
        int gr = m0 + row;
        gr = gr < p.M ? gr : p.M - 1;
        a_off[i] = (unsigned)(gr - m0) * lda + chunk * 16;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int s = i * 256 + tid, row = s >> 2, chunk = (s & 3) ^ ((row >> 2) & 3);
        int gr = c0 + row;
        gr = gr < p.N ? gr : p.N - 1;
        c_off[i] = (unsigned)(gr - c0) * ldw + chunk * 16;
    }
    {
        int gr = c0 + (tid & 127);
        gr = gr < p.N ? gr : p.N - 1;
        q_off = (unsigned)(gr - c0) * (unsigned)G * 2u;
    }
    const unsigned char *a_base = p.x + (long long)m0 * lda;
    const bool second = blockIdx.z != 0;
    const unsigned char *c_base = (second ? p.w2 : p.w) + (long long)c0 * ldw;
    const unsigned short *q_mat = wave < 2 ? (second ? p.scales2 : p.scales) : second ? p.zeros2 : p.zeros;
    const unsigned char *q_base = (const unsigned char *)(q_mat + (long long)c0 * G);
    auto to_lds16 = [&](unsigned char *dst, unsigned off, const unsigned char *src) {
        const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)dst);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
    };
    auto issue = [&](int g, unsigned char *st, int i) {
        if (i < LA) {
            to_lds16(st + (i * 256 + wave * 64) * 16, a_off[i < LA ? i : 0], a_base + (long long)g * 256);
        } else if (i < LA + 2) {
            to_lds16(st + A_BYTES + ((i - LA) * 256 + wave * 64) * 16, c_off[i - LA < 2 ? i - LA : 0], c_base + (long long)g * 64);
        } else {
            const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(st + A_BYTES + kCodeBytes + wave * 256));
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" ::"s"(lds_addr), "v"(q_off), "s"(q_base + (long long)g * 2) : "memory");
        }
    };

    f32x16_t acc[FM];
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[j][q] = 0.f;

    // ---- operands: slice t = 0..7 of a group: step t / 4 (64 k), the lane's 8 k at 64 (t / 4) + 32 h + 8 (t % 4)
    auto read_a = [&](const unsigned char *st, int t, u32x4_t *af) {
        const int chunk = (t >> 2) * 8 + 4 * h + (t & 3);
#pragma unroll
        for (int j = 0; j < FM; ++j)
            af[j] = *reinterpret_cast<const u32x4_t *>(st + (32 * j + r) * 256 + ((chunk ^ (r & 15)) << 4));
    };
    const int crow = 32 * wave + r;
    auto read_codes = [&](const unsigned char *st, u32x4_t *c, float &sc, float &zi, float &rest) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
            c[s] = *reinterpret_cast<const u32x4_t *>(st + A_BYTES + crow * 64 + (((2 * s + h) ^ ((crow >> 2) & 3)) << 4));
        const unsigned *q = reinterpret_cast<const unsigned *>(st + A_BYTES + kCodeBytes);
        const float z = __uint_as_float(q[kCols + crow] << 16);
        sc = __uint_as_float(q[crow] << 16);
        if constexpr (EXACT) {
            lq_split_zero(z, zi, rest);
        } else {  // operands of lq_dequant_word_f32
            zi = -(z * sc);
            sc *= 512.0f;
        }
    };
    auto operand = [](unsigned word, float sc, float zi) {
        if constexpr (EXACT) return lq_codes_minus(word, zi);
        float f[8];
        lq_dequant_word_f32(word, sc, zi, f);
        return u32x4_t{lq_pack_bf16(f[0], f[1]), lq_pack_bf16(f[2], f[3]), lq_pack_bf16(f[4], f[5]), lq_pack_bf16(f[6], f[7])};
    };

    u32x4_t af[2][FM], bf[2], cw[2];
    f32x16_t P[FM];  // EXACT: the group's sums, unscaled
    float sc, zi, rest;
    auto mfma = [](const u32x4_t &a, const u32x4_t &b, const f32x16_t &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    };
    f32x16_t zero;
#pragma unroll
    for (int q = 0; q < 16; ++q) zero[q] = 0.f;
    auto group = [&](int g, auto si) {
        constexpr int S = decltype(si)::value;
        unsigned char *cur = lds + S * STAGE, *nxt = lds + ((S + 1) % D) * STAGE, *fill = lds + ((S + D - 1) % D) * STAGE;
        const int gf = g0 + (g + D - 1 < ng ? g + D - 1 : ng - 1);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const unsigned word_next = t < 7 ? cw[(t + 1) >> 2][(t + 1) & 3] : 0u;
            const float sc_cur = sc;
            if (t == 7) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * LOADS) : "memory");
                read_codes(nxt, cw, sc, zi, rest);
                read_a(nxt, 0, af[0]);
            } else {
                read_a(cur, t + 1, af[(t + 1) & 1]);
                // the loads of the stage the previous group left, spread over the slices
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                    if (i * 7 / LOADS == t) issue(gf, fill, i);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FM; ++j) {
                if constexpr (EXACT) P[j] = mfma(af[t & 1][j], bf[t & 1], t ? P[j] : zero);
                else acc[j] = mfma(af[t & 1][j], bf[t & 1], acc[j]);
            }
            bf[(t + 1) & 1] = operand(t < 7 ? word_next : cw[0][0], sc, zi);
            if constexpr (EXACT) {
                if (t == 6 && __builtin_amdgcn_ballot_w64(rest != 0.0f)) {
                    const u32x4_t b = lq_minus_rest(rest);
#pragma unroll 1
                    for (int v = 0; v < 8; ++v) {
                        u32x4_t a[FM];
                        read_a(cur, v, a);
#pragma unroll
                        for (int j = 0; j < FM; ++j) P[j] = mfma(a[j], b, P[j]);
                    }
                }
                if (t == 7) {
#pragma unroll
                    for (int j = 0; j < FM; ++j)
#pragma unroll
                        for (int q = 0; q < 16; ++q) acc[j][q] = fmaf(sc_cur, P[j][q], acc[j][q]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // prologue: groups 0 .. D - 2
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue(g0 + (d < ng ? d : ng - 1), lds + d * STAGE, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D - 2) * LOADS) : "memory");
    read_codes(lds, cw, sc, zi, rest);
    read_a(lds, 0, af[0]);
    bf[0] = operand(cw[0][0], sc, zi);
    __builtin_amdgcn_sched_barrier(0);
    static_assert(D == 3, "the loop below names the three stages");
    int g = 0;
    for (; g + D <= ng; g += D) {
        group(g, ic<0>());
        group(g + 1, ic<1>());
        group(g + 2, ic<2>());
    }
    if (g < ng) group(g, ic<0>());
    if (g + 1 < ng) group(g + 1, ic<1>());
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the clamped prefetches of the last groups

    // ---- epilogue: acc[j][q]: row m0 + 32 j + 8 (q / 4) + 4 h + q % 4, column c0 + 32 wave + r
    const int c_mine = c0 + 32 * wave + r;
    if (p.partial) {
        float *part = p.partial + (long long)(blockIdx.z * gridDim.y + blockIdx.y) * p.M * p.N;
        if (c_mine < p.N) {
#pragma unroll
            for (int j = 0; j < FM; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    const int m = m0 + 32 * j + 8 * (q >> 2) + 4 * h + (q & 3);
                    if (m < p.M) part[(long long)m * p.N + c_mine] = acc[j][q];
                }
        }
        return;
    }
    __syncthreads();
    constexpr int EP = 80;  // row pitch of the wave's 32 x 32 staging area
    unsigned char *ep = lds + wave * (32 * EP);
    const int ep_row = lane >> 2, ep_chunk = lane & 3;
    const int c_lane = c0 + 32 * wave + ep_chunk * 8;
    const float bias = p.bias && c_mine < p.N ? lq_bf16_bits_to_f32(p.bias[c_mine]) : 0.0f;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
#pragma unroll
        for (int q = 0; q < 16; ++q)
            *reinterpret_cast<unsigned short *>(ep + (8 * (q >> 2) + 4 * h + (q & 3)) * EP + r * 2) =
                lq_f32_to_bf16_bits(p.bias ? acc[j][q] + bias : acc[j][q]);
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int row = it * 16 + ep_row, m = m0 + 32 * j + row;
            const u32x4_t o = *reinterpret_cast<const u32x4_t *>(ep + row * EP + ep_chunk * 16);
            if (m < p.M && c_lane < p.N) *reinterpret_cast<u32x4_t *>(p.y + (long long)m * p.N + c_lane) = o;
        }
    }
    if (p.clk && threadIdx.x == 0) {
        unsigned long long *c = p.clk + 4ll * blockIdx.x;
        c[0] = clk_t0; c[1] = __builtin_amdgcn_s_memtime(); c[2] = clk_r0; c[3] = __builtin_amdgcn_s_memrealtime();
    }
}

template <int FM, bool EXACT>
int launch_staged_tile(StagedParams p, int splits, hipStream_t st, const char *who) {
    p.tiles_m = (p.M + 32 * FM - 1) / (32 * FM);
    p.tiles_n = (p.N + kCols - 1) / kCols;
    const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)splits, p.w2 ? 2u : 1u);
    hipLaunchKernelGGL((gemm_staged_kernel<FM, EXACT>), grid, dim3(256), 0, st, p.x, p.w, p.M, p.N, p.K, p.tiles_m, p.tiles_n, p.groups_per_split,
                       p.scales, p.zeros, p.partial, p.bias, p.y, p.w2, p.scales2, p.zeros2, p.clk);
    return lq_check_launch(who);
}

int launch_staged(const StagedParams &p, int rows, bool exact, int splits, hipStream_t st, const char *who) {
    if (rows == 32) return exact ? launch_staged_tile<1, true>(p, splits, st, who) : launch_staged_tile<1, false>(p, splits, st, who);
    if (rows == 64) return exact ? launch_staged_tile<2, true>(p, splits, st, who) : launch_staged_tile<2, false>(p, splits, st, who);
    return launch_staged_tile<4, false>(p, splits, st, who);
}

}  // namespace

// Row tile and slices of K. The time of a candidate is estimated from its workgroups per compute unit: a group of
// 128 k takes a workgroup 0.45 / 0.54 / 0.74 us with 32 / 64 / 128 rows on an idle device and up to 22 % more with one
// on every unit (clock, HBM); a further resident one (three of 32 rows, two of 64, one of 128 fit) adds 0.30 / 0.46 us,
// plus 0.19 as soon as there is one. 4.1 us around the loop; a split costs 1.7 us for the second launch and 0.53 us per
// MB of partial products. Constants fitted to 2000 timings (12 matrices from 1024^2 to 11008 x 4096, 17 to 1536
// tokens, every row tile, 1 to 8 slices): 5.5 % rms; the choice costs 1.5 % over the best candidate on average.
// A slice has at least four groups.
double lq_gemm_staged_plan(long long M, long long N, int groups, size_t ws_bytes, long long cus, int *rows, int *splits, int *per_split) {
    static const double lone[3] = {0.45, 0.54, 0.74}, more[3] = {0.30, 0.46, 0.0};
    static const int fit_cu[3] = {3, 2, 1};
    const long long cols = (N + kCols - 1) / kCols, tiles128 = (M + 127) / 128 * cols;
    long long most = (long long)(ws_bytes / ((size_t)M * N * 4));
    if (most > cus / tiles128) most = cus / tiles128;
    if (most > 8) most = 8;
    if (most > groups / 4) most = groups / 4;
    double best = 1e30;
    for (int i = 0; i < 3; ++i) {
        const int h = 32 << i;
        if (i && M <= h / 2) continue;  // half of the rows would be padding
        for (int s = 1; s == 1 || s <= most; ++s) {
            const int per = (groups + s - 1) / s;
            if (s > 1 && (per < 4 || (groups + per - 1) / per != s)) continue;
            const double load = (double)((M + h - 1) / h * cols * s) / (double)cus;
            double g = lone[i];
            if (load <= 1.0) g *= 1.0 + 0.22 * load;
            else if (fit_cu[i] == 1) g *= 1.22 * (double)(long long)(load + 0.999);
            else {
                const double res = load < fit_cu[i] ? load : (double)fit_cu[i];
                g = 1.22 * g + (more[i] * (res - 1.0) + 0.19) * (load / res);
            }
            const double est = 4.1 + per * g + (s > 1 ? 1.7 + 0.53e-6 * 4.0 * s * (double)M * (double)N : 0.0);
            if (est < best) { best = est; *rows = h; *splits = s; *per_split = per; }
        }
    }
    return best;
}

// Gate and up product of few tokens as one launch of twice the tiles: fp32 partial products [2][splits][M][N] to `partial`,
// to be added and combined by the caller. Shapes as below; splits >= 1.
int lq_gemm_staged_pair_launch(const void *x, const void *codes_g, const void *scales_g, const void *zeros_g, const void *codes_u,
                               const void *scales_u, const void *zeros_u, float *partial, int M, int N, int K, int rows, int splits,
                               int per_split, hipStream_t st, const char *who) {
    StagedParams p = {};
    p.x = (const unsigned char *)x;
    p.w = (const unsigned char *)codes_g; p.scales = (const unsigned short *)scales_g; p.zeros = (const unsigned short *)zeros_g;
    p.w2 = (const unsigned char *)codes_u; p.scales2 = (const unsigned short *)scales_u; p.zeros2 = (const unsigned short *)zeros_u;
    p.M = M; p.N = N; p.K = K;
    p.partial = partial; p.groups_per_split = per_split;
    return launch_staged(p, rows, false, splits, st, who);
}

// splits > 1: fp32 partial products [splits][M][N] to `partial`, to be added by the caller; else bf16 (x W^T + bias) to y.
// exact: weights not rounded to bf16 (32 or 64 rows). N % 16 == 0, K % 128 == 0, splits == ceil(K / 128 / per_split) are
// guaranteed by the caller.
int lq_gemm_staged_launch(const void *x, const void *codes, const void *scales, const void *zeros, const void *bias, void *y,
                          float *partial, int M, int N, int K, int rows, bool exact, int splits, int per_split, hipStream_t st,
                          unsigned long long *clk, const char *who) {
    StagedParams p = {};
    p.x = (const unsigned char *)x; p.w = (const unsigned char *)codes;
    p.scales = (const unsigned short *)scales; p.zeros = (const unsigned short *)zeros;
    p.bias = (const unsigned short *)bias; p.y = (unsigned short *)y;
    p.M = M; p.N = N; p.K = K; p.clk = clk;
    if (splits > 1) { p.partial = partial; p.groups_per_split = per_split; }
    return launch_staged(p, rows, exact, splits, st, who);
}
