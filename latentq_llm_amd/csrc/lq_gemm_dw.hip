// Weight-gradient GEMM for gfx950:  dW[N,K] = dY[M,N]^T . X[M,K]   (bf16 operands, fp32 accumulation)
//
// The reduction runs over the tokens m, the slow dimension of both operands, so neither operand has the
// layout an MFMA lane wants (8 consecutive reduction elements of one row). Both tiles are staged exactly as they
// lie in memory - 64 token rows of 256 contiguous columns, written by LDS-direct loads (no registers, no
// vector-ALU work) - and the fragments are fetched with the transposing LDS read ds_read_b64_tr_b16: within a
// 16-lane block, lane i receives the four elements of column i of the 4 x 16 block the 16 lanes address. No
// transposed copy of dY is made anywhere.
//
// Three tile sizes (dw_tile below chooses) and two ways through the large one:
//   256 (n) x 256 (k) outputs, 512 threads = 8 waves in a 2 (n) x 4 (k) grid; a wave owns 128 x 64 outputs (4 x 2 MFMA
//     32x32x16 tiles, 128 accumulator registers). Steps of 64 tokens, two LDS stages of 64 KB (64 rows of dY and 64 rows
//     of X, 512 bytes each); one workgroup per CU.
//   the same tile and steps, 256 threads = 2 x 2 waves of 128 x 128 (256 accumulators, one wave per SIMD): 128 instead of
//     192 KB of fragment reads per 64 tokens, which is power the matrix cores get. A lone wave has to issue everything
//     between its own MFMAs, so the reads of the next slice and the loads are dealt out one or two per MFMA, the reads
//     over the first half of a slice, and the whole old gradient is requested before the accumulating epilogue starts. us
//     at 2048 tokens, 8 waves -> 4 (store / accumulate in bf16): 11008 x 4096 172 / 191 -> 157 / 181, 3072^2 49 / 60 -> 45 / 56;
//     4096 tokens, 11008 x 4096 310 / 327 -> 296 / 315. The int8 accumulator's epilogue is vector work that wants two
//     waves (196 -> 211), and with few steps a lone wave's prologue and epilogue show (300 tokens 41 / 64 -> 45 / 71, level
//     at 1024 to 1500): those keep the 8 waves. The sums are taken in the same order, so a gradient stored and then
//     added to an int8 accumulator still has the bits of the fused epilogue. (Steps of 32 tokens in four stages are as
//     fast, but cut a number of tokens that is no multiple of 64 into other slices.)
//   128 x 128 outputs, 256 threads = 2 x 2 waves of 64 x 64. Steps of 32 tokens, four stages of 16 KB, two workgroups
//     per CU: for outputs whose large tiles leave most of the device idle. There a workgroup has nothing but its own
//     prefetch distance to cover its waits, which is what the four stages are for (2048 x 2048 outputs, 2048 tokens:
//     20.4 us against 26.4 with two stages of 64 tokens). Deeper stages gain the large tile nothing (159 against 157 us
//     on 11008 x 4096: it is bound by power, 79 % of the matrix pipe's cycles when few CUs run it).
//
//   192 (n) x 256 (k) outputs in the 8-wave form, 96 x 64 a wave: for outputs of which 256 x 256 tiles leave a third of the CUs idle
//     or begin another round, and 128 x 128 ones pay more ways in and out. 500 tokens, 5504 x 2048 outputs are 172 / 232 large /
//     medium tiles on 256 CUs: 20.0 -> 17.9 us, with the int8 accumulator 26.1 (small tiles) -> 23.9; 1024 tokens, 3072^2 (144 / 192)
//     25.3 -> 22.1 and 32.5 -> 28.0; 2240 tokens, 4736 x 1792 46.2 -> 39.4.
//
// A slice is 16 tokens. Lane l: r = l % 32, h = l / 32; in slice t the lane's operand for column r of a 32-column
// fragment is tokens 16 t + 8 h .. + 7: two transposing reads (tokens .. + 3 and + 4 .. + 7). In each read block lane i
// (of 16) addresses row i / 4 of the block's 4 token rows at columns 4 (i % 4) .. + 3 of its 16 columns. A row is a
// number of 32-byte segments; segment s of token row m sits at position s ^ 2 (m & 3), which spreads the 4 rows x 2
// column blocks that 32 lanes read over all 64 banks (rows of 384 bytes alternate between the halves of the banks by themselves and
// have 12 segments: s ^ (m & 2)); the swizzle is free, since an LDS-direct load lets a lane choose
// the global 16 bytes that land in its slot.
//
// Any number of tokens: see `first` below. Against the tensor library's product, which took the token counts that are
// no multiple of 64 before: 500 tokens, 5504 x 2048 outputs 18.4 against 24.7 us, 1000 tokens, 11008 x 4096 87 against 116.
//
// Pipeline as in the int8 tile kernel: one s_barrier per step before its last slice, loads as inline assembly with
// explicit waits.
//
// D = Xfrag x dYfrag^T: a lane owns 4 consecutive k of one n. Epilogues (through LDS, 16-byte pieces of rows):
//   store  dW rounded to bf16;
//   acc8   the int8 gradient accumulator's add_ form on the bf16-rounded dW: q = quant(dequant(q) + dW) in place
//          with the stored row scale (16 consecutive k per lane = one Philox block), so that neither dW nor the
//          dequantised accumulator ever exists in memory.
#include "lq_common.h"
#include "lq_gradq8_math.h"

#include <type_traits>

namespace {

struct DwParams {
    const unsigned char *dy;  // bf16 [M, N]
    const unsigned char *x;   // bf16 [M, K]
    unsigned short *dw;       // store: bf16 [N, K]
    int accumulate;           // store: dw = bf16(dw + bf16(product)) instead of dw = bf16(product)
    signed char *q;           // acc8: int8 [N, K], updated in place
    const unsigned short *scale;  // acc8: bf16 [N]
    const unsigned short *noise;  // acc8: bf16 [N, K] or null (Philox)
    unsigned long long seed, offset;
    int M, N, K;
    int tiles_n, tiles_k;
};

typedef __attribute__((address_space(3))) void lds_void;
typedef short v4s_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v4s_t lds_v4s_t;

template <int I>
using ic = std::integral_constant<int, I>;

// TILE_N, TILE_K: outputs per workgroup, NT: its threads. STEP_M: tokens per reduction step; NST: LDS stages of one step.
template <int TILE_N, int TILE_K, int NT, int STEP_M, int NST, bool ACC8>
__global__ __launch_bounds__(NT) void gemm_dw_kernel(DwParams p) {
    constexpr int ROW_A = TILE_N * 2, ROW_B = TILE_K * 2;  // bytes per staged token row of dY, of X
    constexpr int A_STAGE = STEP_M * ROW_A, STAGE = A_STAGE + STEP_M * ROW_B;
    constexpr int LA = A_STAGE / 16 / NT, LB = STEP_M * ROW_B / 16 / NT;  // 16-byte loads per thread and stage
    constexpr int SL = STEP_M / 16;            // slices of a step (an even number)
    constexpr int WM = 2, WN = NT / 64 / WM;       // waves along n, along k
    constexpr int TM = TILE_N / WM, TN = TILE_K / WN;  // wave tile: 128 n x 64 k, 96 x 64, or 64 x 64
    constexpr int FM = TM / 32, FN = TN / 32;
    constexpr bool kLone = FM * FN == 16;  // 256 accumulators: one wave per SIMD
    static_assert(!kLone || !ACC8, "the int8 epilogue wants two waves per SIMD");
    // the stages; the accumulate epilogue stages every wave's whole block (144-byte rows) instead
    constexpr int EP_ALL = WM * WN * TM * (TN * 2 + 16);
    constexpr int LDS_BYTES = ACC8 && EP_ALL > NST * STAGE ? EP_ALL : NST * STAGE;
    __shared__ __attribute__((aligned(16))) unsigned char lds_all[LDS_BYTES];
    auto stage = [&](int i) -> unsigned char * { return lds_all + (i % NST) * STAGE; };

    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int r = lane & 31, h = lane >> 5;
    const int wm = wave % WM, wn = wave / WM;

    // Workgroup ids are dealt round-robin over the 8 XCDs (id % 8): give each XCD a contiguous range of the tile
    // sequence, ordered in bands of GN tile columns walked row by row, so the workgroups resident on one XCD share
    // a few dY column blocks and X column blocks in its L2.
    const int nwg = p.tiles_n * p.tiles_k;
    int id = blockIdx.x;
    {
        const int per = nwg / 8;
        if (id < per * 8) id = (id % 8) * per + id / 8;
    }
    constexpr int GN = 8;
    const int band = id / (p.tiles_n * GN);
    const int within = id - band * (p.tiles_n * GN);
    const int rest = p.tiles_k - band * GN;
    const int bw = rest < GN ? rest : GN;
    const int tile_n = within / bw, tile_k = band * GN + within % bw;
    const int n0 = tile_n * TILE_N, k0 = tile_k * TILE_K;
    // A number of tokens that is no multiple of the step leaves the FIRST step short: its last rows are tokens 0 .. first - 1
    // (the rows ahead of them re-read the last of these and are masked out of both operands), and every later step starts on
    // a full stride. Counted from the end the tokens then fall into the same slices of 16 whatever the step, so that the tile
    // sizes add in one order and the store and accumulate forms agree in every bit where they take different ones.
    const int nk = (p.M + STEP_M - 1) / STEP_M;
    const int first = p.M - (nk - 1) * STEP_M;

    // ---- staging: slot s = i * NT + thread of an operand's stage is token row s / (TILE / 8), 16-byte position
    // s % (TILE / 8); it receives the 16 bytes of segment (pos / 2) ^ flip(row), half pos & 1. Columns past the end of a matrix
    // re-read its last 8 columns (their results are dropped).
    auto flip = [](int row, int row_bytes) { return row_bytes % 256 == 0 ? 2 * (row & 3) : row & 2; };
    unsigned a_off[LA], b_off[LB];
    auto offset = [&](int i, int tile, int first_col, int cols) {
        const int s = i * NT + (int)threadIdx.x;
        const int row = s / (tile / 8), pos = s % (tile / 8);
        const int c = first_col / 8 + ((((pos >> 1) ^ flip(row, tile * 2)) << 1) | (pos & 1));
        return (unsigned)((long long)row * cols * 2 + (long long)(c < cols / 8 ? c : cols / 8 - 1) * 16);
    };
#pragma unroll
    for (int i = 0; i < LA; ++i) a_off[i] = offset(i, TILE_N, n0, p.N);
#pragma unroll
    for (int i = 0; i < LB; ++i) b_off[i] = offset(i, TILE_K, k0, p.K);
    // load i of a step: 0 .. LA - 1 fill the dY rows of the stage, the LB others its X rows
    auto issue_off = [&](long long row0, unsigned char *st, int i, unsigned off) {
        const bool is_b = i >= LA;
        const int ii = is_b ? i - LA : i;
        const unsigned char *src = is_b ? p.x + row0 * p.K * 2 : p.dy + row0 * p.N * 2;
        const unsigned lds_addr = (unsigned)reinterpret_cast<size_t>(
            (lds_void *)(st + (is_b ? A_STAGE : 0) + (ii * NT + wave * 64) * 16));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds_addr), "v"(off), "s"(src) : "memory");
    };
    auto issue_one = [&](int kt, unsigned char *st, int i) {  // kt >= 1, or a full first step
        issue_off((long long)kt * STEP_M - (STEP_M - first), st, i, i >= LA ? b_off[i >= LA ? i - LA : 0] : a_off[i < LA ? i : 0]);
    };
    auto issue_first = [&](unsigned char *st, int i) {  // step 0: rows ahead of token 0 read the step's last token
        const int row = ((i >= LA ? i - LA : i) * NT + (int)threadIdx.x) / ((i >= LA ? TILE_K : TILE_N) / 8), ahead = STEP_M - first;
        const unsigned back = (unsigned)(row >= ahead ? ahead : row - (first - 1));  // (modulo 2^32: the offsets stay within the step's tokens)
        issue_off(0, st, i, i >= LA ? b_off[i >= LA ? i - LA : 0] - back * (unsigned)(p.K * 2) : a_off[i < LA ? i : 0] - back * (unsigned)(p.N * 2));
    };

    // ---- fragments. Read block = lane / 16: column block (lane / 16) & 1 of the fragment's 32 columns, token half
    // h; block lane i16 addresses token row (i16 / 4) of the block's 4 and columns 4 (i16 % 4) .. + 3.
    const int i16 = lane & 15, cblk = (lane >> 4) & 1;
    // byte offset of the lane's 8 bytes within a staged row of fragment f (32 columns from column 32 f of the wave's part)
    auto col_off = [&](int col0, int row_bytes) {
        const int seg = (col0 >> 4) + cblk;  // 32-byte segment of the row
        return ((seg ^ flip(i16 >> 2, row_bytes)) << 5) + ((i16 & 3) << 3);
    };
    int a_col[FM], b_col[FN];
#pragma unroll
    for (int j = 0; j < FM; ++j) a_col[j] = col_off(wm * TM + 32 * j, ROW_A);
#pragma unroll
    for (int i = 0; i < FN; ++i) b_col[i] = A_STAGE + col_off(wn * TN + 32 * i, ROW_B);
    const int row_a = (8 * h + (i16 >> 2)) * ROW_A, row_b = (8 * h + (i16 >> 2)) * ROW_B;  // + 16 t rows for slice t, + 4 rows for the second read
    // a short first step: the lane's rows 16 t + 8 h + e of slice t ahead of the first token become zero
    auto mask_frag = [&](u32x4_t &f, int t) {
        const int ahead = STEP_M - first - (16 * t + 8 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const unsigned keep = ahead <= 2 * e ? 0xFFFFFFFFu : ahead == 2 * e + 1 ? 0xFFFF0000u : 0u;
            f[e] &= keep;
        }
    };
    // half e (tokens .. + 3, .. + 7) of fragment f of slice t: dY fragments 0 .. FM - 1, then X fragments
    auto read_half = [&](const unsigned char *st, int t, u32x4_t *af, u32x4_t *bf, int f, int e) {
        const unsigned char *base = st + (f < FM ? row_a + (t * 16 + 4 * e) * ROW_A : row_b + (t * 16 + 4 * e) * ROW_B);
        const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s_t *)(base + (f < FM ? a_col[f < FM ? f : 0] : b_col[f >= FM ? f - FM : 0]))));
        u32x4_t &d = f < FM ? af[f < FM ? f : 0] : bf[f >= FM ? f - FM : 0];
        d[2 * e] = v[0];
        d[2 * e + 1] = v[1];
    };
    auto read_frags = [&](const unsigned char *st, int t, u32x4_t *af, u32x4_t *bf) {
#pragma unroll
        for (int f = 0; f < FM + FN; ++f) {
            read_half(st, t, af, bf, f, 0);
            read_half(st, t, af, bf, f, 1);
        }
    };

    f32x16_t acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.f;

    u32x4_t af[2][FM], bf[2][FN];
    auto mfma_slice = [&](const u32x4_t *a, const u32x4_t *b) {
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
            for (int j = 0; j < FM; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, b[i]),
                                                                   __builtin_bit_cast(bf16x8_t, a[j]), acc[i][j], 0, 0, 0);
    };
    // Step kt: the operands of its first slice are already in af[0] / bf[0]. The barrier stands before the last slice: it
    // finds step kt + 1 landed (all but the loads of the steps after it), every wave's reads of this step returned, and
    // releases this step's stage. The last slice then reads the first operands of step kt + 1 and issues the dY half of
    // step kt + NST into the stage just released; the next step's first slice issues the X half.
    auto step = [&](int kt, auto si, auto masked) {
        constexpr int S = decltype(si)::value;                 // the step's stage
        constexpr bool MASKED = decltype(masked)::value != 0;  // the short first step
        unsigned char *cur = stage(S), *nxt = stage(S + 1), *left = stage(S + NST - 1);
        // (the last steps re-load the last step's rows)
        const int kt_x = kt + NST - 1 < nk ? kt + NST - 1 : nk - 1, kt_dy = kt + NST < nk ? kt + NST : nk - 1;
        auto load = [&](int k, unsigned char *st, int i) {
            if (MASKED && k == 0) issue_first(st, i);
            else issue_one(k, st, i);
        };
#pragma unroll
        for (int t = 0; t < SL; ++t) {
            if (t == SL - 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NST - 2) * (LA + LB)) : "memory");
            const unsigned char *src = t < SL - 1 ? cur : nxt;
            const int tn = t < SL - 1 ? t + 1 : 0;
            if constexpr (kLone && !MASKED) {
                // one wave per SIMD: everything else is dealt out between the MFMAs, the reads of the next slice (in the
                // order in which it uses them) over the first half of them, so that they are back when it starts
                static_assert(FM == FN && LA == LB && LA <= FM * FN, "one load per MFMA at most");
#pragma unroll
                for (int m = 0; m < FM * FN; ++m) {
                    constexpr int kReads = 2 * (FM + FN), kPer = kReads / (FM * FN / 2);
#pragma unroll
                    for (int q = 0; q < kPer; ++q) {
                        const int n = m * kPer + q;  // halves: dY 0, X 0, dY 1, X 1, ...
                        if (n < kReads) read_half(src, tn, af[tn & 1], bf[tn & 1], (n >> 1) % 2 == 0 ? (n >> 2) : FM + (n >> 2), n & 1);
                    }
                    if (m % 2 == 1 && m / 2 < LA) {
                        if (t == 0) load(kt_x, left, LA + m / 2);
                        if (t == SL - 1) load(kt_dy, cur, m / 2);
                    }
                    const int i = m / FM, j = m % FM;
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, bf[t & 1][i]),
                                                                       __builtin_bit_cast(bf16x8_t, af[t & 1][j]), acc[i][j], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                continue;
            }
            read_frags(src, tn, af[tn & 1], bf[tn & 1]);
            if (t == 0) {
#pragma unroll
                for (int i = LA; i < LA + LB; ++i) load(kt_x, left, i);
            }
            if (t == SL - 1) {
#pragma unroll
                for (int i = 0; i < LA; ++i) load(kt_dy, cur, i);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (MASKED) {
#pragma unroll
                for (int j = 0; j < FM; ++j) mask_frag(af[t & 1][j], t);
#pragma unroll
                for (int i = 0; i < FN; ++i) mask_frag(bf[t & 1][i], t);
            }
            mfma_slice(af[t & 1], bf[t & 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // prologue: steps 0 .. NST - 2 and the dY half of step NST - 1; wait for step 0. A short first step takes the last
    // stage, so that the loop below starts on stage 0 either way.
    const int shift = first < STEP_M ? NST - 1 : 0;
#pragma unroll
    for (int s = 0; s < NST; ++s)
#pragma unroll
        for (int i = 0; i < (s == NST - 1 ? LA : LA + LB); ++i) {
            const int k = s < nk ? s : nk - 1;
            if (k == 0) issue_first(stage(s + shift), i);
            else issue_one(k, stage(s + shift), i);
        }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NST - 2) * (LA + LB) + LA) : "memory");
    read_frags(stage(shift), 0, af[0], bf[0]);
    __builtin_amdgcn_sched_barrier(0);
    int kt = 0;
    if (first < STEP_M) step(kt++, ic<NST - 1>(), ic<1>());
    for (; kt + NST <= nk; kt += NST) {
        step(kt, ic<0>(), ic<0>());
        step(kt + 1, ic<1>(), ic<0>());
        if constexpr (NST > 2) step(kt + 2, ic<2 % NST>(), ic<0>());
        if constexpr (NST > 3) step(kt + 3, ic<3 % NST>(), ic<0>());
    }
    static_assert(NST <= 4, "the loop above has up to four steps");
    const int rem = nk - kt;
    if (rem > 0) step(kt, ic<0>(), ic<0>());
    if constexpr (NST > 2) if (rem > 1) step(kt + 1, ic<1>(), ic<0>());
    if constexpr (NST > 3) if (rem > 2) step(kt + 2, ic<2 % NST>(), ic<0>());
    // the clamped prefetches of the last steps are still writing LDS: drain them
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- epilogue: acc[i][j][q]: column k0 + TN wn + 32 i + 8 (q / 4) + 4 h + q % 4, row n0 + TM wm + 32 j + r.
    // Every wave passes its block through a private LDS area.
    __syncthreads();
    constexpr int EP = TN * 2 + 16;  // row pitch of the staging area
    const int kw0 = k0 + wn * TN;
    if constexpr (!ACC8) {
        // 32 rows (one j) at a time; 16 bytes per lane, TN / 8 lanes on the contiguous bytes of a row
        unsigned char *ep = lds_all + wave * (32 * EP);
        constexpr int LPR = TN / 8, RPI = 64 / LPR;
        const int ep_row = lane / LPR, ep_chunk = lane % LPR;
        const int kc = kw0 + ep_chunk * 8;
        constexpr int IT = 32 / RPI;
        unsigned short *const out = p.dw + (long long)(n0 + wm * TM + ep_row) * p.K + kc;
        auto live = [&](int j, int it) { return n0 + wm * TM + j * 32 + it * RPI + ep_row < p.N && kc < p.K; };
        auto piece = [&](int j, int it) { return reinterpret_cast<u32x4_t *>(out + (long long)(j * 32 + it * RPI) * p.K); };
        auto emit = [&](auto accumulate) {
            constexpr bool ACC = decltype(accumulate)::value != 0;
            // The old gradient of the rows ahead: a lone wave has no other to cover the latency, and its fragments' registers
            // are free by now, so it asks for the whole block at once; two waves per SIMD take 32 rows at a time.
            constexpr int AHEAD = kLone ? FM : 1;
            u32x4_t old[ACC ? AHEAD : 1][IT];
            auto fetch = [&](int j) {
#pragma unroll
                for (int it = 0; it < IT; ++it) {
                    old[ACC ? j % AHEAD : 0][it] = u32x4_t{0u, 0u, 0u, 0u};
                    if (live(j, it)) old[ACC ? j % AHEAD : 0][it] = *piece(j, it);
                }
            };
            if constexpr (ACC && AHEAD > 1) {
#pragma unroll
                for (int j = 0; j < FM; ++j) fetch(j);
            }
#pragma unroll
            for (int j = 0; j < FM; ++j) {
                if constexpr (ACC && AHEAD == 1) fetch(j);
#pragma unroll
                for (int i = 0; i < FN; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const u32x2_t o = {lq_pack_bf16(acc[i][j][4 * q], acc[i][j][4 * q + 1]), lq_pack_bf16(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3])};
                        *reinterpret_cast<u32x2_t *>(ep + r * EP + (i * 32 + 8 * q + 4 * h) * 2) = o;
                    }
#pragma unroll
                for (int it = 0; it < IT; ++it) {
                    u32x4_t o = *reinterpret_cast<const u32x4_t *>(ep + (it * RPI + ep_row) * EP + ep_chunk * 16);
                    if constexpr (ACC) {
                        // the bf16 addition a tensor `add_` of the stored product would make
                        const u32x4_t g = old[j % AHEAD][it];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            o[e] = lq_pack_bf16(lq_bf16_lo(g[e]) + lq_bf16_lo(o[e]), lq_bf16_hi(g[e]) + lq_bf16_hi(o[e]));
                    }
                    if (live(j, it)) *piece(j, it) = o;
                }
            }
        };
        if (p.accumulate) emit(ic<1>());
        else emit(ic<0>());
    } else {
        // The whole block of the wave goes to LDS as bf16 first (straight-line code), then a rolled loop of
        // TM / RPP passes of 16 rows does the accumulator arithmetic: unrolled over the accumulator registers that
        // arithmetic would be some 50 KB of code, more than the instruction cache holds. 16 consecutive k per lane
        // (one Philox block), 4 lanes per row.
        unsigned char *ep = lds_all + wave * (TM * EP);
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const u32x2_t o = {lq_pack_bf16(acc[i][j][4 * q], acc[i][j][4 * q + 1]), lq_pack_bf16(acc[i][j][4 * q + 2], acc[i][j][4 * q + 3])};
                    *reinterpret_cast<u32x2_t *>(ep + (j * 32 + r) * EP + (i * 32 + 8 * q + 4 * h) * 2) = o;
                }
        constexpr int PPR = TN / 16, RPP = 64 / PPR;  // pieces per row, rows per pass
        const int q_row = lane / PPR, q_piece = lane % PPR;
        const int kq = kw0 + q_piece * 16;
        const int nw0 = n0 + wm * TM;
        auto fetch = [&](int pass, u32x4_t &oldq, float &sc) {
            const int nn = nw0 + pass * RPP + q_row;
            const bool live = nn < p.N && kq < p.K;
            oldq = *reinterpret_cast<const u32x4_t *>(p.q + (live ? (long long)nn * p.K + kq : 0));
            sc = lq_bf16_bits_to_f32(p.scale[live ? nn : 0]);
        };
        u32x4_t old_next;
        float s_next;
        fetch(0, old_next, s_next);
#pragma unroll 1
        for (int pass = 0; pass < TM / RPP; ++pass) {
            const u32x4_t oldq = old_next;
            const float sc = s_next;
            if (pass + 1 < TM / RPP) fetch(pass + 1, old_next, s_next);
            const int row = pass * RPP + q_row;
            const int nn = nw0 + row;
            const bool live = nn < p.N && kq < p.K;
            const u32x4_t v0 = *reinterpret_cast<const u32x4_t *>(ep + row * EP + q_piece * 32);
            const u32x4_t v1 = *reinterpret_cast<const u32x4_t *>(ep + row * EP + q_piece * 32 + 16);
            const long long e0 = live ? (long long)nn * p.K + kq : 0;
            u32x4_t z0 = {0u, 0u, 0u, 0u}, z1 = z0;
            if (p.noise) {
                z0 = *reinterpret_cast<const u32x4_t *>(p.noise + e0);
                z1 = *reinterpret_cast<const u32x4_t *>(p.noise + e0 + 8);
            }
            const unsigned long long c = p.offset + (unsigned long long)(e0 >> 4);
            // the reciprocal form is exact for scales between 2^-40 and 2^40; one lane outside sends the wave
            // through the division
            const bool fast = sc >= 0x1p-40f && sc <= 0x1p40f;
            const bool all_fast = __builtin_amdgcn_ballot_w64(!fast) == 0ull;
            u32x4_t o;
            if (p.noise) o = all_fast ? quant16<false, true, true>(v0, v1, oldq, z0, z1, sc, 1.0f / sc, c, p.seed)
                                      : quant16<false, true, false>(v0, v1, oldq, z0, z1, sc, 0.f, c, p.seed);
            else o = all_fast ? quant16<true, true, true>(v0, v1, oldq, z0, z1, sc, 1.0f / sc, c, p.seed)
                              : quant16<true, true, false>(v0, v1, oldq, z0, z1, sc, 0.f, c, p.seed);
            if (live) *reinterpret_cast<u32x4_t *>(p.q + e0) = o;
        }
    }
}

template <int TILE_N, int TILE_K, int NT, int STEP_M, int NST, bool ACC8>
static int launch_dw_tile(DwParams p, hipStream_t st, const char *who) {
    p.tiles_n = (p.N + TILE_N - 1) / TILE_N;
    p.tiles_k = (p.K + TILE_K - 1) / TILE_K;
    const long long nwg = (long long)p.tiles_n * p.tiles_k;
    if (nwg > 0x7FFFFFFFll) return lq_fail(LQ_ERR_BAD_ARG, "%s: problem too large", who);
    // the 32-bit lane offsets of the loads span a step's token rows
    if (64ll * 2 * (p.N > p.K ? p.N : p.K) >= (1ll << 32)) return lq_fail(LQ_ERR_BAD_ARG, "%s: rows too long", who);
    const dim3 grid((unsigned)nwg), block(NT);
    hipLaunchKernelGGL((gemm_dw_kernel<TILE_N, TILE_K, NT, STEP_M, NST, ACC8>), grid, block, 0, st, p);
    return lq_check_launch(who);
}

// Which tile a product takes: the smallest of three estimates in microseconds, all of the form (time per 64-token step, summed
// over the rounds of workgroups) x steps + the ways in and out. The last round is never empty: 256 tiles on 256 CUs are one full "last"
// round. A round of large tiles steps more slowly with more than half of the CUs busy (power), one of 128 x 128 tiles as the
// second workgroup of a CU joins. What comes around the steps depends on the form: bf16 stores, a gradient read and added as well, or the
// int8 accumulator's arithmetic, some 17 instructions an element, which want every CU and another workgroup's steps beside
// them; the four-wave form has steps and ways of its own. us, 128 x 128 / 192 x 256 / 256 x 256:
//   tokens, outputs     2048, 2048^2   2000, 8192 x 3072   500, 8192 x 3072   500, 5504 x 2048     64, 4096 x 1536   2000, 11008 x 4096
//   store               20.4 / - / 39.8    94.9 / - / 92.6     32.2 / 40.4 / 34.1   19.9 / 17.9 / 20.0   6.5 / - / 7.7     171 / - / 153
//   int8                23.9 / - / 51.0    105 / - / 115       43.8 / 60.7 / 52.8   26.1 / 23.9 / 32.1   11.3 / - / 17.4   188 / - / 186
// The constants are fitted to 2500 products (8 to 4096 tokens, 768^2 to 11008 x 4096) timed in each form with each tile: to the times
// (off by 5 % on average), but above all to the choice, which costs 0.19 / 0.13 / 0.02 % (store, add, int8) over the fastest tile. Against the
// choice between 128 x 128 and 256 x 256 by one estimate for all forms it takes 0.968 / 0.962 / 0.936 of the time, 18 products of the
// 7500 are more than 2 % slower (at most 9), and 7 of 1500 that it was not fitted to (at most 7). Constants with one set for both
// 256 x 256 forms and nothing for a masked step had 108 of the 7500: 13 tokens, 4096^2 store 11.9 against 10.9; 3316, 3584 x 11008 add 262 against 242; 64, 3584 x 8832 int8 41.5 against 39.1. Level
// tiles are not told apart: 65 to 95 tokens, 11008 x 4096 store 28.8 against 27.7, 4096 x 11008 28.5 against 29.1.
enum DwForm { DW_STORE, DW_ACC, DW_ACC8 };
enum DwTile { DW_128, DW_192, DW_256, DW_256_LONE };

static DwTile dw_tile(DwForm form, long long M, long long N, long long K, long long cus) {
    struct Step { double full, last, busy, ragged; };  // us per step of a full round, of the last one, and more by the share of the CUs beyond
                                                       // half; a masked first step, per round
    struct Ways { double once, round, share; };        // us per launch, per full round, by the last one's share of the CUs
    constexpr Step kStep256 = {1.727, 1.002, 0.733, 0.173}, kStepLone = {1.313, 1.009, 1.076, 0.344}, kStep192 = {1.297, 0.806, 0.672, 0.227};
    constexpr Ways kWays256[] = {{5.592, 7.523, 3.459}, {8.216, 16.138, 6.378}, {15.406, 19.057, 4.035}};
    constexpr Ways kWaysLone[] = {{5.195, 12.784, 3.316}, {4.709, 22.364, 10.903}};
    constexpr Ways kWays192[] = {{3.873, 6.196, 3.281}, {8.216, 12.575, 4.083}, {11.188, 14.900, 5.485}};
    constexpr Ways kWays128[] = {{3.967, 3.740, 1.090}, {4.001, 7.607, 4.524}, {7.150, 8.756, 1.542}};
    constexpr double kSecond[] = {1.024, 2.759, 4.916};  // 128 x 128: once more, where CUs have two workgroups
    const double steps = (double)((M + 63) / 64);
    // one workgroup to a compute unit
    auto whole = [&](long long tiles, const Step &s, const Ways &w) {
        const long long rounds = (tiles - 1) / cus;
        const double share = (double)(tiles - rounds * cus) / (double)cus;  // the last round's share of the CUs, 0 .. 1
        const double step = s.full * (double)rounds + s.last + (share > 0.5 ? s.busy * (share - 0.5) : 0.0);
        return step * steps + w.once + w.round * (double)rounds + w.share * share + (M % 64 ? s.ragged * (double)(rounds + 1) : 0.0);
    };
    // 4 waves of 128 x 128 from where their faster steps outweigh the longer way in and out (see the top of the file)
    const bool lone = form != DW_ACC8 && M >= 1536;
    const long long tiles_k = (K + 255) / 256, t128 = ((N + 127) / 128) * ((K + 127) / 128);
    const double est256 = whole((N + 255) / 256 * tiles_k, lone ? kStepLone : kStep256, lone ? kWaysLone[form] : kWays256[form]);
    const double est192 = whole((N + 191) / 192 * tiles_k, kStep192, kWays192[form]);
    const long long rounds128 = (t128 - 1) / (2 * cus);
    const double r128 = (double)(t128 - rounds128 * 2 * cus) / (double)cus;  // 0 .. 2 workgroups per CU
    const double step128 = 0.858 * (double)rounds128 + (r128 <= 1 ? 0.355 + 0.204 * r128 : 0.745 + 0.049 * (r128 - 1));
    const Ways &w128 = kWays128[form];
    const double est128 = step128 * 0.5 * (double)((M + 31) / 32) + w128.once + w128.round * (double)rounds128 +
                          (r128 <= 1 ? w128.share * r128 : kSecond[form] + w128.share * (r128 - 1)) +
                          (M % 32 ? 0.185 * (double)(rounds128 + 1) : 0.0);
    const double large = est192 < est256 ? est192 : est256;
    return est128 < large ? DW_128 : est192 < est256 ? DW_192 : lone ? DW_256_LONE : DW_256;
}

static int launch_dw(const DwParams &p, DwForm form, hipStream_t st, const char *who) {
    const DwTile tile = dw_tile(form, p.M, p.N, p.K, lq_device_cu_count());
    if (form == DW_ACC8)
        return tile == DW_128   ? launch_dw_tile<128, 128, 256, 32, 4, true>(p, st, who)
               : tile == DW_192 ? launch_dw_tile<192, 256, 512, 64, 2, true>(p, st, who)
                                : launch_dw_tile<256, 256, 512, 64, 2, true>(p, st, who);
    return tile == DW_128   ? launch_dw_tile<128, 128, 256, 32, 4, false>(p, st, who)
           : tile == DW_192 ? launch_dw_tile<192, 256, 512, 64, 2, false>(p, st, who)
           : tile == DW_256 ? launch_dw_tile<256, 256, 512, 64, 2, false>(p, st, who)
                            : launch_dw_tile<256, 256, 256, 64, 2, false>(p, st, who);
}

static int check_dw_sizes(const char *who, int64_t M, int64_t N, int64_t K, int k_mult) {
    LQ_REQUIRE(M > 0 && N > 0 && K > 0 && M < (1ll << 31) && N < (1ll << 31) && K < (1ll << 31), "%s: M, N, K must be positive", who);
    LQ_REQUIRE(N % 8 == 0 && K % k_mult == 0, "%s: N=%lld must be a multiple of 8 and K=%lld of %d", who, (long long)N, (long long)K, k_mult);
    return LQ_OK;
}

static int check_dw(const char *who, const void *dy, const void *x, int64_t M, int64_t N, int64_t K, int k_mult) {
    LQ_REQUIRE(dy && x, "%s: null pointer argument", who);
    const int rc = check_dw_sizes(who, M, N, K, k_mult);
    if (rc) return rc;
    LQ_REQUIRE(lq_aligned(dy, 16) && lq_aligned(x, 16), "%s: dy and x must be 16-byte aligned", who);
    return LQ_OK;
}

}  // namespace

extern "C" int lq_weight_grad_plan(int form, int64_t M, int64_t N, int64_t K, int compute_units, int *rows, int *columns, int *waves) {
    LQ_REQUIRE(rows && columns && waves, "lq_weight_grad_plan: null pointer argument");
    LQ_REQUIRE(form >= DW_STORE && form <= DW_ACC8, "lq_weight_grad_plan: form=%d must be 0, 1 or 2", form);
    int rc = check_dw_sizes("lq_weight_grad_plan", M, N, K, form == DW_ACC8 ? 16 : 8);
    if (rc) return rc;
    const DwTile tile = dw_tile((DwForm)form, M, N, K, compute_units > 0 ? compute_units : lq_device_cu_count());
    *rows = tile == DW_128 ? 128 : tile == DW_192 ? 192 : 256;
    *columns = tile == DW_128 ? 128 : 256;
    *waves = tile == DW_128 || tile == DW_256_LONE ? 4 : 8;
    return LQ_OK;
}

extern "C" int lq_weight_grad(const void *dy, const void *x, void *dw_out, int64_t M, int64_t N, int64_t K, void *stream) {
    int rc = check_dw("lq_weight_grad", dy, x, M, N, K, 8);
    if (rc) return rc;
    LQ_REQUIRE(dw_out && lq_aligned(dw_out, 16), "lq_weight_grad: dw_out must be given, 16-byte aligned");
    DwParams p = {};
    p.dy = (const unsigned char *)dy; p.x = (const unsigned char *)x; p.dw = (unsigned short *)dw_out;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    return launch_dw(p, DW_STORE, (hipStream_t)stream, "lq_weight_grad");
}

extern "C" int lq_weight_grad_acc(const void *dy, const void *x, void *dw_inout, int64_t M, int64_t N, int64_t K, void *stream) {
    int rc = check_dw("lq_weight_grad_acc", dy, x, M, N, K, 8);
    if (rc) return rc;
    LQ_REQUIRE(dw_inout && lq_aligned(dw_inout, 16), "lq_weight_grad_acc: dw_inout must be given, 16-byte aligned");
    DwParams p = {};
    p.dy = (const unsigned char *)dy; p.x = (const unsigned char *)x; p.dw = (unsigned short *)dw_inout;
    p.accumulate = 1;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    return launch_dw(p, DW_ACC, (hipStream_t)stream, "lq_weight_grad_acc");
}

extern "C" int lq_weight_grad_acc8(const void *dy, const void *x, int8_t *q_inout, const void *scale, int64_t M, int64_t N,
                                   int64_t K, const void *noise_or_null, uint64_t philox_seed, uint64_t philox_offset,
                                   void *stream) {
    int rc = check_dw("lq_weight_grad_acc8", dy, x, M, N, K, 16);
    if (rc) return rc;
    LQ_REQUIRE(q_inout && scale && lq_aligned(q_inout, 16) && lq_aligned(scale, 2) && (!noise_or_null || lq_aligned(noise_or_null, 16)),
               "lq_weight_grad_acc8: q and scale must be given; q and noise 16-byte aligned");
    DwParams p = {};
    p.dy = (const unsigned char *)dy; p.x = (const unsigned char *)x; p.q = (signed char *)q_inout;
    p.scale = (const unsigned short *)scale; p.noise = (const unsigned short *)noise_or_null;
    p.seed = philox_seed; p.offset = philox_offset;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    return launch_dw(p, DW_ACC8, (hipStream_t)stream, "lq_weight_grad_acc8");
}
