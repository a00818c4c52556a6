// Forward GEMM of the A16W4 layers with both operands staged in LDS, for grids of few workgroups:
//   Y[M,N] = X[M,K] . deq(W)[N,K]^T (+ bias), the fp32 partial products of slices of K, or h = silu(X Wg^T) * (X Wu^T)
//
// 17 to some 500 tokens: a compute unit gets one workgroup, so nothing hides a load behind another workgroup's work and the
// time is that of the serial chain through one workgroup's slice of K. What the kernel does about it:
//   * LDS-direct loads three stages deep: two stages of loads are in flight while one is multiplied, with one barrier per stage;
//   * codes stay packed in LDS and each wave converts the 32 columns it multiplies, in registers: no second trip through LDS
//     and no waves that only convert;
//   * eight waves, two for each 32 columns, that work on different k and add up at the end: a wave alone on its SIMD issues
//     its MFMAs, conversions and LDS reads one behind the other (128 rows and a long slice of K, or
//     rows of an odd number of groups: four, see gemm_staged_four_kernel);
//   * whole cache lines: what a unit takes in through L1 (30 bytes a clock with all units asking) counts in lines of 128
//     bytes. Codes come in pieces of 128 bytes of a row, two groups of 128 k; scales and zeros 16 bytes at a time;
//   * a plain product of up to 64 tokens (128 without a workspace) does not round its weights to bf16, since the GEMV, which
//     ran many of these sizes before, does not either: the operand is the integer q - rint(z), exact in bf16, and the scale is
//     applied in fp32 to the sum of a group. Zeros that are no integers of at most 240 add a second product with the
//     remainder (`rest` below). Against the weights as they are a result is 1.66e-3 off, its own rounding, instead of 2.22e-3;
//   * the row tile is 32, 64 or 128 tokens, so that few tokens are not mostly padding; the planner below picks it
//     together with the number of slices of K;
//   * a gate / up product whose K is not cut takes 64 columns of both matrices into a workgroup and writes h itself.
// Bound: vector instructions up to 64 rows (19 per 8 weights and lane, 600 cycles per SIMD and group of 128 k for a tile's 128
// columns: 0.3 of the 0.44 / 0.51 us a group takes; with every load answered by L2 the loop is no faster), LDS reads beside
// MFMAs with 128 (one 16-byte fragment read per MFMA).
// Measured, weights from HBM, us: before (four waves, a group of 128 k per stage, a 2-byte scale load per column and group, a
// second launch for h) -> now
//     plain N x K     17 tokens       45              64              100            384
//     4096 x 11008    16.9 -> 16.4    19.4 -> 18.7    20.0 -> 19.2    24.2 -> 24.2
//     4096 x 4096                                                                    26.0 -> 23.6
//     11008 x 4096                    21.0 -> 18.6
//     32000 x 4096    26.2 -> 22.8 (32 tokens)        32.4 -> 27.9 (60)
//     h: 11008 x 4096 25.3 -> 19.4    29.3 -> 23.2    30.4 -> 23.5    41.5 -> 36 (128)
//     h: 6144 x 3072                                                  25.0 -> 18.5
//     h: 4096 x 2048                                                  21.2 -> 14.3 (200)
#include "lq_common.h"
#include "lq_staged_ring.h"

#include <type_traits>

namespace {

struct StagedParams {
    const unsigned char *x;  // bf16 [M, K]
    const unsigned char *w;  // packed codes
    const unsigned short *scales, *zeros, *bias;
    // a second matrix of the same shape on the same activations, or null: both give partial products (blockIdx.z = 1 the
    // second's), or h
    const unsigned char *w2;
    const unsigned short *scales2, *zeros2;
    unsigned short *y;       // bf16 [M, N]; gate / up: h
    unsigned short *g_out, *u_out;  // gate / up: the two products, or null
    float *partial;          // partial products: fp32 [matrices][splits][M][N], or null
    int M, N, K;
    int tiles_m, tiles_n;
    int groups_per_split;    // groups of 128 k per slice (blockIdx.y)
    int q_log;               // log2 of the groups in a piece of scales and zeros: 3, 2 or 0
    unsigned long long *clk; // measurement aid, see lq_calib_gemm_clocks; null in normal use
};

typedef __attribute__((address_space(3))) void lds_void;

template <int I>
using ic = std::integral_constant<int, I>;

constexpr int kCols = 128;
constexpr int kThreads = 512;
// LDS stages; a fourth changes nothing, with two the 128-row tile takes 15 % longer
constexpr int D = kStagedStages;

// LDS (every 16-byte piece swizzled so that the fragment reads, one piece of 32 consecutive rows, spread over all banks).
// FM < 4: a stage is a pair of groups (256 k); of the two waves on a column block one multiplies the first group, one the second.
//   activations  32 FM rows of 512 bytes, chunk c of row i at c ^ (i & 15)
//   codes        128 rows of 128 bytes,   chunk c of row i at c ^ ((i >> 1) & 7)
// FM = 4, for which that is too much: a stage is one group, of which each wave takes 64 k
//   activations  128 rows of 256 bytes,   chunk c of row i at c ^ (i & 15)
//   codes        as above, a pair of groups in one of two slots, requested every other stage
// Scales and zeros: a ring of pieces (lq_staged_ring.h), see issue_q.
constexpr int kCodeBytes = kCols * 128;

// FM: 32-row fragments of the row tile (32 FM rows)
// EXACT: weights as they are (see the top of the file), else rounded to bf16 like those of the kernels for more tokens
// GU: columns 0 .. 63 of the tile are rows of the first matrix, 64 .. 127 the same rows of the second
// Arguments: those of the first loads first (the leading 14 dwords are preloaded into registers, build.py)
template <int FM, bool EXACT, bool GU>
__global__ __launch_bounds__(kThreads, 2) void gemm_staged_kernel(
    const unsigned char *x_, const unsigned char *w_, int M, int N, int K, int tiles_m, int tiles_n, int groups_per_split,
    int q_log, const unsigned short *scales, const unsigned short *zeros, float *partial, const unsigned short *bias_, unsigned short *y,
    const unsigned char *w2, const unsigned short *scales2, const unsigned short *zeros2, unsigned short *g_out, unsigned short *u_out,
    unsigned long long *clk) {
    const StagedParams p = {x_, w_, scales, zeros, bias_, w2, scales2, zeros2, y, g_out, u_out, partial, M, N, K, tiles_m, tiles_n,
                            groups_per_split, q_log, clk};
    constexpr bool PAIRS = FM < 4;
    constexpr int BM = 32 * FM;
    constexpr int A_ROW = PAIRS ? 512 : 256, A_BYTES = BM * A_ROW;
    constexpr int C_SLOTS = PAIRS ? D : 2;
    constexpr int SLICES = PAIRS ? 8 : 4;             // slices of 16 k (8 per lane half) a wave multiplies per stage
    constexpr int LA = A_BYTES / 16 / kThreads;       // loads per thread and stage: activations
    constexpr int LC = kCodeBytes / 16 / kThreads;    // codes (FM = 4: every other stage)
    constexpr int EP = 136;                           // floats per row of the sums in LDS (4 rows apart: 32 banks)
    constexpr int LDS_BYTES = D * A_BYTES + C_SLOTS * kCodeBytes + ScaleRing::bytes(PAIRS);
    static_assert(2 * BM * EP * 4 <= LDS_BYTES, "the sums do not fit");
    static_assert(PAIRS || !EXACT, "128 rows: rounded weights only");
    __shared__ __attribute__((aligned(16))) unsigned char lds[LDS_BYTES];
    unsigned char *const lds_c = lds + D * A_BYTES, *const q_ring = lds_c + C_SLOTS * kCodeBytes;

    const int wave_all = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int kg = wave_all >> 2, wave = wave_all & 3;
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
    const int m0 = tile_m * BM, c0 = tile_n * (GU ? kCols / 2 : kCols);
    const int G = p.K / LQ_GROUP;
    const int g_first = p.partial ? (int)blockIdx.y * p.groups_per_split : 0;
    const int g_end = p.partial && g_first + p.groups_per_split < G ? g_first + p.groups_per_split : G;
    const StagedSlice slice = {g_first, g_end, PAIRS};
    const ScaleRing ring = {p.q_log, PAIRS};
    const int units = slice.units(), my_units = slice.units_of(kg);
    const int half_of_one = G == 1 ? 1 : 0;                 // a row of one group: both halves of a pair are that group

    // ---- loads
    unsigned a_off[LA], c_off[LC];
    const unsigned lda = (unsigned)p.K * 2u, ldw = (unsigned)p.K / 2u;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int s = i * kThreads + tid, row = s / (A_ROW / 16);
        int chunk = (s % (A_ROW / 16)) ^ (row & 15);
        if (PAIRS && half_of_one) chunk &= 15;
        int gr = m0 + row;
        gr = gr < p.M ? gr : p.M - 1;
        a_off[i] = (unsigned)(gr - m0) * lda + chunk * 16;
    }
    auto tile_row = [&](int i) {  // row of its matrix, from c0, that is column i of the tile
        const int row = GU ? i & 63 : i;
        return c0 + row < p.N ? row : p.N - 1 - c0;
    };
#pragma unroll
    for (int i = 0; i < LC; ++i) {
        const int s = i * kThreads + tid, row = s >> 3;
        int chunk = (s & 7) ^ ((row >> 1) & 7);
        if (half_of_one) chunk &= 3;
        c_off[i] = (unsigned)tile_row(row) * ldw + chunk * 16;
    }
    const unsigned char *a_base = p.x + (long long)m0 * lda;
    const bool second = !GU && blockIdx.z != 0;
    const unsigned char *c_base = (second ? p.w2 : p.w) + (long long)c0 * ldw, *c_base2 = GU ? p.w2 + (long long)c0 * ldw : c_base;
    auto scalar = [](const unsigned char *q) {  // the loads take their base from scalar registers
        const unsigned long long a = (unsigned long long)q;
        return (const unsigned char *)(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
                                       (unsigned)__builtin_amdgcn_readfirstlane((int)a));
    };
    auto to_lds16 = [&](unsigned char *dst, unsigned off, const unsigned char *from) {
        const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)dst);
        const unsigned char *src = scalar(from);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
    };
    auto issue_a = [&](int u, unsigned char *st, int i) {
        const int g = slice.group_of(u, 0);
        to_lds16(st + (i * kThreads + wave_all * 64) * 16, a_off[i], a_base + (long long)g * 256);
    };
    static_assert(LC == 2, "gate / up: the first load of the codes is the first matrix', the second the second's");
    auto issue_c = [&](int j, unsigned char *slot, int i) {
        to_lds16(slot + (i * kThreads + wave_all * 64) * 16, c_off[i], (i ? c_base2 : c_base) + (long long)slice.pair_start(j) * 64);
    };
    // Scales and zeros of 2^q_log groups in a piece, fetched by the first four waves: 16 bytes per column, 8 values from an even
    // index on: 8 groups, or 4 of rows of an odd number of groups, which may begin at the second value. The last piece
    // ends with the matrix. q_log = 0, matrices that are not 4-byte aligned: one value, in a dword. A slot holds
    // [scales, zeros][128 columns].
    const int q_most = (p.N - c0 < kCols ? p.N - c0 : kCols) * G - 8;
    const unsigned q_shift = p.q_log ? 4u : 2u;
    auto q_first = [&](int row_at, int piece) {  // index of a piece's first value, for the row that begins at index row_at
        const int at = row_at + (piece << p.q_log);
        if (!p.q_log) return at;
        return (at & ~1) < q_most ? at & ~1 : q_most;
    };
    const unsigned short *q_mat = GU ? (wave & 1 ? (wave < 2 ? p.scales2 : p.zeros2) : wave < 2 ? p.scales : p.zeros)
                                     : wave < 2 ? (second ? p.scales2 : p.scales) : second ? p.zeros2 : p.zeros;
    const unsigned char *q_base = scalar((const unsigned char *)(q_mat + (long long)c0 * G));
    const int q_row = tile_row(tid & 127) * G;
    int q_next = ring.piece(g_first);  // pieces below have been requested
    auto issue_q = [&](int g) {        // all pieces up to group g's; whether this wave issued any
        const bool any = kg == 0 && q_next <= ring.piece(g);
        for (; q_next <= ring.piece(g); ++q_next) {
            if (kg) continue;
            const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(q_ring + ((ring.slot(q_next) * 256 + wave * 64) << q_shift)));
            const unsigned off = (unsigned)q_first(q_row, q_next) * 2u;
            if (p.q_log) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(q_base) : "memory");
            else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_ushort %1, %2" ::"s"(lds_addr), "v"(off), "s"(q_base) : "memory");
        }
        return any;
    };

    f32x16_t acc[FM];
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[j][q] = 0.f;

    // ---- operands: slice t = 0..7 of a group: step t / 4 (64 k), the lane's 8 k at 64 (t / 4) + 32 h + 8 (t % 4)
    // (FM = 4: t = 0..3, the step is the wave's)
    auto read_a = [&](const unsigned char *st, int t, u32x4_t *af) {
        const int chunk = (PAIRS ? kg * 16 + (t >> 2) * 8 : kg * 8) + 4 * h + (t & 3);
#pragma unroll
        for (int j = 0; j < FM; ++j)
            af[j] = *reinterpret_cast<const u32x4_t *>(st + (32 * j + r) * A_ROW + ((chunk ^ (r & 15)) << 4));
    };
    const int crow = 32 * wave + r, crow_q = tile_row(crow) * G;
    // where a stage's codes and its scale (the zero: kCols entries behind) are in LDS
    int c_at[SLICES / 4], q_at;
    auto find_codes = [&](int u, int stage) {
        const int start = slice.pair_start(PAIRS ? u : u >> 1), g = slice.group_of(u, kg);
        const int half = PAIRS ? kg : g - start, slot = (PAIRS ? stage : (u >> 1) & 1) * kCodeBytes;
#pragma unroll
        for (int s = 0; s < SLICES / 4; ++s) {
            const int chunk = 4 * half + (PAIRS ? 2 * s : 2 * kg) + h;
            c_at[s] = slot + crow * 128 + ((chunk ^ ((crow >> 1) & 7)) << 4);
        }
        const int gq = g < g_end ? g : g_end - 1, piece = ring.piece(gq);
        q_at = (int)((ring.slot(piece) * 256 + crow) << q_shift) + (crow_q + gq - q_first(crow_q, piece)) * 2;
    };
    auto read_codes = [&](u32x4_t *c, float &sc, float &zi, float &rest) {
        sc = lq_bf16_bits_to_f32(*reinterpret_cast<const unsigned short *>(q_ring + q_at));
        const float z = lq_bf16_bits_to_f32(*reinterpret_cast<const unsigned short *>(q_ring + q_at + (kCols << q_shift)));
#pragma unroll
        for (int s = 0; s < SLICES / 4; ++s) c[s] = *reinterpret_cast<const u32x4_t *>(lds_c + c_at[s]);
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

    u32x4_t af[2][FM], bf[2], cw[SLICES / 4];
    f32x16_t P[FM];  // EXACT: the group's sums, unscaled
    float sc, zi, rest;
    auto mfma = [](const u32x4_t &a, const u32x4_t &b, const f32x16_t &c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    };
    f32x16_t zero;
#pragma unroll
    for (int q = 0; q < 16; ++q) zero[q] = 0.f;
    auto code_slot = [&](int u, int stage) { return lds_c + (PAIRS ? stage : (u >> 1) & 1) * kCodeBytes; };
    // this wave's part of the next stage has landed: all but the loads of the last stage requested
    auto wait_and_meet = [](auto n, bool piece) {
        constexpr int N = (D - 2) * decltype(n)::value;
        if (piece) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N + 1) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
    };
    // keeps what is computed under one slice's MFMAs there: the compiler moves it behind the next branch otherwise
    auto stays = [](auto &&v) { asm volatile("" : "+v"(v)); };
    auto stage = [&](int u, auto si) {
        constexpr int S = decltype(si)::value;
        unsigned char *cur = lds + S * A_BYTES, *nxt = lds + ((S + 1) % D) * A_BYTES, *fill = lds + ((S + D - 1) % D) * A_BYTES;
        const int uf = u + D - 1 < units ? u + D - 1 : units - 1;
        const bool codes_too = PAIRS || !(u & 1), piece = u + D - 1 < units && issue_q(slice.last_group(uf));
#pragma unroll
        for (int t = 0; t < SLICES; ++t) {
            const unsigned word_next = t < SLICES - 1 ? cw[(t + 1) >> 2][(t + 1) & 3] : 0u;
            const float sc_cur = sc;
            if (t == SLICES - 1) {
                if (codes_too) wait_and_meet(ic<LA + LC>(), piece);
                else wait_and_meet(ic<LA>(), piece);
                read_codes(cw, sc, zi, rest);
                read_a(nxt, 0, af[0]);
            } else {
                read_a(cur, t + 1, af[(t + 1) & 1]);
                // the loads of the stage the previous one left, spread over the slices
#pragma unroll
                for (int i = 0; i < LA + LC; ++i)
                    if (i * (SLICES - 1) / (LA + LC) == t) {
                        if (i >= LC) issue_a(uf, fill, i - LC);
                        else if (codes_too) issue_c(PAIRS ? uf : uf >> 1, code_slot(u + D - 1, (S + D - 1) % D), i);
                    }
                if (t == SLICES - 2) {
                    find_codes(u + 1, (S + 1) % D);
#pragma unroll
                    for (int s = 0; s < SLICES / 4; ++s) stays(c_at[s]);
                    stays(q_at);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < FM; ++j) {
                if constexpr (EXACT) P[j] = mfma(af[t & 1][j], bf[t & 1], t ? P[j] : zero);
                else acc[j] = mfma(af[t & 1][j], bf[t & 1], acc[j]);
            }
            if (t == SLICES - 1) __builtin_amdgcn_sched_barrier(0);  // the products before the wait for the next codes
            bf[(t + 1) & 1] = operand(t < SLICES - 1 ? word_next : cw[0][0], sc, zi);
            stays(bf[(t + 1) & 1]);
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

    // prologue: stages 0 .. D - 2
    static_assert(D == 3, "the prologue and the loop below name the three stages");
    issue_q(slice.last_group(0));
#pragma unroll
    for (int i = 0; i < LC; ++i) issue_c(0, code_slot(0, 0), i);
#pragma unroll
    for (int i = 0; i < LA; ++i) issue_a(0, lds, i);
    const int u1 = units > 1 ? 1 : 0;
    if (u1) issue_q(slice.last_group(1));
    if constexpr (PAIRS)
#pragma unroll
        for (int i = 0; i < LC; ++i) issue_c(u1, code_slot(1, 1), i);
#pragma unroll
    for (int i = 0; i < LA; ++i) issue_a(u1, lds + A_BYTES, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PAIRS ? LA + LC : LA) : "memory");
    find_codes(0, 0);
    read_codes(cw, sc, zi, rest);
    read_a(lds, 0, af[0]);
    bf[0] = operand(cw[0][0], sc, zi);
    __builtin_amdgcn_sched_barrier(0);
    int u = 0;
    for (; u + D <= my_units; u += D) {
        stage(u, ic<0>());
        stage(u + 1, ic<1>());
        stage(u + 2, ic<2>());
    }
    if (u < my_units) stage(u, ic<0>());
    if (u + 1 < my_units) stage(u + 1, ic<1>());
    if (my_units < units) asm volatile("s_barrier" ::: "memory");  // every wave meets as many barriers
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");               // the clamped prefetches of the last stages
    __syncthreads();

    // ---- epilogue: acc[j][q]: row 32 j + 8 (q / 4) + 4 h + q % 4, column 32 wave + r. Both waves' sums to LDS, from where
    // they are added and leave as 16 bytes per lane.
    float *const sums = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int j = 0; j < FM; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q) sums[(kg * BM + 32 * j + 8 * (q >> 2) + 4 * h + (q & 3)) * EP + crow] = acc[j][q];
    __syncthreads();
    auto sum4 = [&](int row, int c) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t *>(sums + row * EP + c);
        const f32x4_t b = *reinterpret_cast<const f32x4_t *>(sums + (BM + row) * EP + c);
        return f32x4_t{a[0] + b[0], a[1] + b[1], a[2] + b[2], a[3] + b[3]};
    };
    auto pack8 = [](const float *v) {
        return u32x4_t{lq_pack_bf16(v[0], v[1]), lq_pack_bf16(v[2], v[3]), lq_pack_bf16(v[4], v[5]), lq_pack_bf16(v[6], v[7])};
    };
    if (!GU && p.partial) {
        float *part = p.partial + (long long)(blockIdx.z * gridDim.y + blockIdx.y) * p.M * p.N;
        for (int i = tid; i < BM * (kCols / 4); i += kThreads) {
            const int row = i / (kCols / 4), c = i % (kCols / 4) * 4;
            if (m0 + row < p.M && c0 + c < p.N) *reinterpret_cast<f32x4_t *>(part + (long long)(m0 + row) * p.N + c0 + c) = sum4(row, c);
        }
        return;
    }
    constexpr int CPR = (GU ? kCols / 2 : kCols) / 8;  // 16-byte pieces of a result row
    for (int i = tid; i < BM * CPR; i += kThreads) {
        const int row = i / CPR, c = i % CPR * 8;
        if (m0 + row >= p.M || c0 + c >= p.N) continue;
        const long long at = (long long)(m0 + row) * p.N + c0 + c;
        float v[8], o[8];
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const f32x4_t a = sum4(row, c + e);
#pragma unroll
            for (int k = 0; k < 4; ++k) v[e + k] = a[k];
        }
        if constexpr (GU) {
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; e += 4) {
                const f32x4_t a = sum4(row, kCols / 2 + c + e);
#pragma unroll
                for (int k = 0; k < 4; ++k) w[e + k] = a[k];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = v[e] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[e])) * w[e];
            *reinterpret_cast<u32x4_t *>(p.y + at) = pack8(o);
            if (p.g_out) {
                *reinterpret_cast<u32x4_t *>(p.g_out + at) = pack8(v);
                *reinterpret_cast<u32x4_t *>(p.u_out + at) = pack8(w);
            }
        } else {
            if (p.bias) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] += lq_bf16_bits_to_f32(p.bias[c0 + c + e]);
            }
            *reinterpret_cast<u32x4_t *>(p.y + at) = pack8(v);
        }
    }
    if (p.clk && threadIdx.x == 0) {
        unsigned long long *c = p.clk + 4ll * blockIdx.x;
        c[0] = clk_t0; c[1] = __builtin_amdgcn_s_memtime(); c[2] = clk_r0; c[3] = __builtin_amdgcn_s_memrealtime();
    }
}

// 128-row tiles on four waves of 32 columns, a group of 128 k per stage, codes in pieces of 64 bytes, scales
// and zeros 2 bytes at a time. Where the loop is long the kernel above is the slower one: its two waves on a column block wait
// for each other at every barrier without filling each other's gaps, since LDS reads beside MFMAs fill them already; and where
// rows are an odd number of groups, or a slice begins at an odd one, its 128-byte pieces of codes lie across two cache lines. us,
// weights from HBM, eight waves -> four:
//   in one line  4096 x 11008 at 1019 tokens 100.3 -> 97.8, 2560 x 8192 at 1500 72.4 -> 70.8
//   across two   3840 x 9088 at 632 69.7 -> 64.5, 2816 x 10880 at 876 81.8 -> 72.8, 7808 x 1408 at 336 14.7 -> 14.0; two slices: 3840 x 11008 at 370 54.6 -> 51.1,
//                6272 x 7936 at 245 43.8 -> 39.4
// LDS of a stage, swizzled like the one above:
//   activations  128 rows of 256 bytes, chunk c of row i at c ^ (i & 15)
//   codes        128 rows of 64 bytes,  chunk c of row i at c ^ ((i >> 2) & 3)
//   scales, zeros  one dword per column each, the bf16 value in its lower half
constexpr int kFourThreads = 256;
__global__ __launch_bounds__(kFourThreads) void gemm_staged_four_kernel(StagedParams p) {
    constexpr int FM = 4, BM = 32 * FM, A_BYTES = BM * 256, C_BYTES = kCols * 64, STAGE = A_BYTES + C_BYTES + kCols * 8;
    constexpr int LA = A_BYTES / 16 / kFourThreads, LC = C_BYTES / 16 / kFourThreads;
    constexpr int LOADS = LA + LC + 1;  // per thread and stage: activations, codes, one scale or zero
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
    const int tile_m = id % p.tiles_m, tile_n = id / p.tiles_m;
    const int m0 = tile_m * BM, c0 = tile_n * kCols;
    const int G = p.K / LQ_GROUP;
    const int g0 = p.partial ? (int)blockIdx.y * p.groups_per_split : 0;
    const int g1 = p.partial && g0 + p.groups_per_split < G ? g0 + p.groups_per_split : G;
    const int ng = g1 - g0;

    // ---- loads
    unsigned a_off[LA], c_off[LC];
    const unsigned lda = (unsigned)p.K * 2u, ldw = (unsigned)p.K / 2u;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int s = i * kFourThreads + tid, row = s >> 4, chunk = (s & 15) ^ (row & 15);
        a_off[i] = (unsigned)((m0 + row < p.M ? m0 + row : p.M - 1) - m0) * lda + chunk * 16;
    }
    auto tile_row = [&](int row) { return (unsigned)(c0 + row < p.N ? row : p.N - 1 - c0); };
#pragma unroll
    for (int i = 0; i < LC; ++i) {
        const int s = i * kFourThreads + tid, row = s >> 2, chunk = (s & 3) ^ ((row >> 2) & 3);
        c_off[i] = tile_row(row) * ldw + chunk * 16;
    }
    const unsigned q_off = tile_row(tid & 127) * (unsigned)G * 2u;
    const unsigned char *a_base = p.x + (long long)m0 * lda, *c_base = p.w + (long long)c0 * ldw;
    const unsigned char *q_base = (const unsigned char *)((wave < 2 ? p.scales : p.zeros) + (long long)c0 * G);
    auto to_lds16 = [&](unsigned char *dst, unsigned off, const unsigned char *src) {
        const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)dst);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(off), "s"(src) : "memory");
    };
    auto issue = [&](int g, unsigned char *st, int i) {
        if (i < LA) {
            to_lds16(st + (i * kFourThreads + wave * 64) * 16, a_off[i < LA ? i : 0], a_base + (long long)g * 256);
        } else if (i < LA + LC) {
            to_lds16(st + A_BYTES + ((i - LA) * kFourThreads + wave * 64) * 16, c_off[i - LA < LC ? i - LA : 0], c_base + (long long)g * 64);
        } else {
            const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>((lds_void *)(st + A_BYTES + C_BYTES + wave * 256));
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
    auto read_codes = [&](const unsigned char *st, u32x4_t *c, float &sc, float &zs) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
            c[s] = *reinterpret_cast<const u32x4_t *>(st + A_BYTES + crow * 64 + (((2 * s + h) ^ ((crow >> 2) & 3)) << 4));
        const unsigned *q = reinterpret_cast<const unsigned *>(st + A_BYTES + C_BYTES);
        sc = __uint_as_float(q[crow] << 16);
        zs = -(__uint_as_float(q[kCols + crow] << 16) * sc);  // operands of lq_dequant_word_f32
        sc *= 512.0f;
    };
    auto operand = [](unsigned word, float sc, float zs) {
        float f[8];
        lq_dequant_word_f32(word, sc, zs, f);
        return u32x4_t{lq_pack_bf16(f[0], f[1]), lq_pack_bf16(f[2], f[3]), lq_pack_bf16(f[4], f[5]), lq_pack_bf16(f[6], f[7])};
    };

    u32x4_t af[2][FM], bf[2], cw[2];
    float sc, zs;
    auto group = [&](int g, auto si) {
        constexpr int S = decltype(si)::value;
        unsigned char *cur = lds + S * STAGE, *nxt = lds + ((S + 1) % D) * STAGE, *fill = lds + ((S + D - 1) % D) * STAGE;
        const int gf = g0 + (g + D - 1 < ng ? g + D - 1 : ng - 1);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const unsigned word_next = t < 7 ? cw[(t + 1) >> 2][(t + 1) & 3] : 0u;
            if (t == 7) {
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((D - 2) * LOADS) : "memory");
                read_codes(nxt, cw, sc, zs);
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
            for (int j = 0; j < FM; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, af[t & 1][j]),
                                                                 __builtin_bit_cast(bf16x8_t, bf[t & 1]), acc[j], 0, 0, 0);
            bf[(t + 1) & 1] = operand(t < 7 ? word_next : cw[0][0], sc, zs);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // prologue: groups 0 .. D - 2
    static_assert(D == 3, "the loop below names the three stages");
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
#pragma unroll
        for (int i = 0; i < LOADS; ++i) issue(g0 + (d < ng ? d : ng - 1), lds + d * STAGE, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((D - 2) * LOADS) : "memory");
    read_codes(lds, cw, sc, zs);
    read_a(lds, 0, af[0]);
    bf[0] = operand(cw[0][0], sc, zs);
    __builtin_amdgcn_sched_barrier(0);
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
        float *part = p.partial + (long long)blockIdx.y * p.M * p.N;
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

// Whether a slice of so many groups goes to four waves in 128-row tiles: where it is long, and sooner where the other kernel's
// pieces of codes, two groups, lie across cache lines (rows of an odd number of groups; slices that begin at an odd one), the more
// so the fewer row tiles read the codes after the first. Speed of four waves over eight, medians over 3500 sizes (1024 to 8192
// columns, 65 to 2048 tokens, every slice the planner cuts):
//     groups of the slice                 6-17   18-23  24-31  32-41  42-49  50-59  60-71  72-95  96-
//     pieces in one line                  0.964  0.970  0.977  0.980  0.99   0.998  1.014  1.022  1.025
//     across two, K whole                 1.013  1.006  1.006  1.010  1.020  1.04   1.055  1.076  1.10
//     across two, K cut, 2 row tiles      0.982  1.013  1.026  1.04
//                        3                0.972  0.985  1.008  1.024  1.04
//                        4 and more       0.972  0.980  0.988  1.002  1.011  1.036
constexpr bool four_waves(int groups_of_row, int groups_of_slice, int row_tiles) {
    const bool whole = groups_of_slice >= groups_of_row, across = groups_of_row % 2 || (!whole && groups_of_slice % 2);
    return groups_of_slice >= (!across ? 60 : whole ? 0 : row_tiles <= 2 ? 18 : row_tiles == 3 ? 25 : 32);
}

int launch_staged_four(StagedParams p, int splits, hipStream_t st, const char *who) {
    p.tiles_m = (p.M + 127) / 128;
    p.tiles_n = (p.N + kCols - 1) / kCols;
    hipLaunchKernelGGL(gemm_staged_four_kernel, dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)splits), dim3(kFourThreads), 0, st, p);
    return lq_check_launch(who);
}

template <int FM, bool EXACT, bool GU>
int launch_staged_tile(StagedParams p, int splits, hipStream_t st, const char *who) {
    const int cols = GU ? kCols / 2 : kCols;
    p.tiles_m = (p.M + 32 * FM - 1) / (32 * FM);
    p.tiles_n = (p.N + cols - 1) / cols;
    const uintptr_t at = (uintptr_t)p.scales | (uintptr_t)p.zeros | (uintptr_t)p.scales2 | (uintptr_t)p.zeros2;
    p.q_log = at % 4 ? 0 : p.K / LQ_GROUP % 2 ? 2 : 3;
    const dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)splits, !GU && p.w2 ? 2u : 1u);
    hipLaunchKernelGGL((gemm_staged_kernel<FM, EXACT, GU>), grid, dim3(kThreads), 0, st, p.x, p.w, p.M, p.N, p.K, p.tiles_m, p.tiles_n,
                       p.groups_per_split, p.q_log, p.scales, p.zeros, p.partial, p.bias, p.y, p.w2, p.scales2, p.zeros2, p.g_out, p.u_out, p.clk);
    return lq_check_launch(who);
}

int launch_staged(const StagedParams &p, int rows, bool exact, int splits, hipStream_t st, const char *who) {
    if (p.w2 && !p.partial)
        return rows == 32   ? launch_staged_tile<1, false, true>(p, 1, st, who)
               : rows == 64 ? launch_staged_tile<2, false, true>(p, 1, st, who)
                            : launch_staged_tile<4, false, true>(p, 1, st, who);
    if (rows == 32) return exact ? launch_staged_tile<1, true, false>(p, splits, st, who) : launch_staged_tile<1, false, false>(p, splits, st, who);
    if (rows == 64) return exact ? launch_staged_tile<2, true, false>(p, splits, st, who) : launch_staged_tile<2, false, false>(p, splits, st, who);
    if (!p.w2 && four_waves(p.K / LQ_GROUP, p.partial ? p.groups_per_split : p.K / LQ_GROUP, (p.M + 127) / 128))
        return launch_staged_four(p, splits, st, who);
    return launch_staged_tile<4, false, false>(p, splits, st, who);
}

}  // namespace

// Row tile and slices of K. The time of a candidate is estimated from its workgroups per compute unit: a group of
// 128 k takes a workgroup 0.45 / 0.54 / 0.74 us with 32 / 64 / 128 rows on an idle device and up to 22 % more with one
// on every unit (clock, HBM); from two on the units' rounds of them (`more`: what each of up to `rounds` adds). 4.1 us
// around the loop; a split costs 1.7 us for the second launch and 0.53 us per MB of partial products. On 730 timings (10
// matrices from 2048^2 to 11008 x 4096, 17 to 1019 tokens, every row tile, 1 to 8 slices) the choice costs 1.2 % over the
// best candidate on average; constants fitted to those timings (0.44 / 0.51 / 0.80 us, 2.4 us) 0.9 %.
// A slice has at least four groups.
double lq_gemm_staged_plan(long long M, long long N, int groups, size_t ws_bytes, long long cus, int *rows, int *splits, int *per_split) {
    static const double lone[3] = {0.45, 0.54, 0.74}, more[3] = {0.30, 0.46, 0.0};
    static const int rounds[3] = {3, 2, 1};
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
            else if (rounds[i] == 1) g *= 1.22 * (double)(long long)(load + 0.999);
            else {
                const double res = load < rounds[i] ? load : (double)rounds[i];
                g = 1.22 * g + (more[i] * (res - 1.0) + 0.19) * (load / res);
            }
            const double est = 4.1 + per * g + (s > 1 ? 1.7 + 0.53e-6 * 4.0 * s * (double)M * (double)N : 0.0);
            if (est < best) { best = est; *rows = h; *splits = s; *per_split = per; }
        }
    }
    return best;
}

// Gate and up product of few tokens. splits = 1: one launch that writes h (and g and u unless null). Otherwise one launch of
// twice the tiles: fp32 partial products [2][splits][M][N] to `partial`, to be added and combined by the caller.
int lq_gemm_staged_pair_launch(const void *x, const void *codes_g, const void *scales_g, const void *zeros_g, const void *codes_u,
                               const void *scales_u, const void *zeros_u, void *h, void *g_out, void *u_out, float *partial, int M, int N,
                               int K, int rows, int splits, int per_split, hipStream_t st, const char *who) {
    StagedParams p = {};
    p.x = (const unsigned char *)x;
    p.w = (const unsigned char *)codes_g; p.scales = (const unsigned short *)scales_g; p.zeros = (const unsigned short *)zeros_g;
    p.w2 = (const unsigned char *)codes_u; p.scales2 = (const unsigned short *)scales_u; p.zeros2 = (const unsigned short *)zeros_u;
    p.M = M; p.N = N; p.K = K;
    if (splits > 1) {
        p.partial = partial; p.groups_per_split = per_split;
    } else {
        p.y = (unsigned short *)h; p.g_out = (unsigned short *)g_out; p.u_out = (unsigned short *)u_out;
    }
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
