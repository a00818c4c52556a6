// Int8 product of few tokens for gfx950:
//   Y[M,N] = bf16(((int32) X8[M,K] . W8[N,K]^T) * sx[m] * sw[n] (+ bias)),  M <= 32
//
// Bound: latency. The weights of a layer (2 to 64 MB) are read once and nothing is reused but the few rows of X, so
// a launch lasts as long as its longest chain of loads. A workgroup owns 16 output columns; its 8 waves share K in units
// of 128 (a cache line of every weight row) and load the 16-byte pieces an MFMA 16x16x64 lane needs straight into
// registers, no LDS and no barrier in between; the eight partial sums meet in LDS once at the end. 128 x 128 tiles, which
// ran these products before, give N / 128 workgroups a serial chain of K / 128 steps.
//
// Up to 16 tokens in inference the activations come in as bf16 and every workgroup quantises all of them itself into
// LDS (kFused; M (K + 16) bytes, at most 64 KB: 16 elements per thread for 4 tokens of 2048): that replaces the
// quantiser's launch or two in front of the product, each of which costs more than the work. The first weight pieces are
// requested behind the activations and travel meanwhile.
//
// MFMA operands: weights first, activations second, so that lane l holds columns 4 (l / 16) .. + 3 of token l % 16.
// In a unit u the lane's pieces are the 16 bytes at k = 128 u + 64 t + 16 (l / 16), t = 0, 1, of row l % 16.
#include "lq_common.h"
#include "lq_actq_math.h"

namespace {

struct Gemv8Params {
    const unsigned short *xf;    // kFused: bf16 [M, K]
    const unsigned char *x8;     // else int8 [M, K]
    const float *sx;             // and fp32 [M]
    const unsigned char *w;      // int8 [N, K]
    const void *sw;              // [N]: fp32, or bf16 when sw_bf16 is set
    int sw_bf16;
    int per_token;               // kFused: one scale per token (else the tensor's maximum is the clamp value)
    const unsigned short *bias;  // bf16 [N] or null
    int *acc_out;                // optional int32 [M, N]
    unsigned short *y;           // bf16 [M, N]
    int M, N, K;
    unsigned row_inv;            // kFused: ceil(2^32 / (K / 8)), the pieces of a token row
};

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kFusedLds = 64 << 10;
constexpr int kDeep = 4096;  // from this K on a wave has four units to request at once; before, the surplus only costs

// FM: groups of 16 tokens. UB: units a wave has in flight. PT: pieces of 8 activations a thread holds (kFused, one scale
// for the tensor): they are requested at once and quantised from registers. Half of them in a loop that read them again
// cost two more round trips to L2 each time: 12.2 us instead of 10.9 on 2048 x 8192 at 4 tokens. Every unit quantises all
// activations, so their instructions count: maxima over pairs of elements and across lanes in registers, no look at each
// element for NaNs (their maximum shows them) took 184 instructions for 8 elements to 95. us: 4 tokens, 2048 x 2048 4.53 ->
// 3.96, 8192 x 2048 6.85 -> 5.94, 2048 x 8192 11.67 -> 9.70; 15 tokens, 1536 x 1536 6.86 -> 5.38, per token 7.79 -> 6.89.
// Arguments: those of the first loads first, the leading 14 dwords are preloaded into registers (build.py): 4 tokens, 8192 x 2048
// 6.91 -> 6.62 us.
template <int FM, bool kFused, int UB, int PT = 1>
__global__ __launch_bounds__(kThreads) void gemv_i8_kernel(const void *x, const unsigned char *w, int M, int N, int K, unsigned row_inv, int per_token,
                                                           int sw_bf16, const void *sw, const unsigned short *bias, unsigned short *y,
                                                           const float *sx, int *acc_out) {
    const Gemv8Params p = {(const unsigned short *)x, (const unsigned char *)x, sx, w, sw, sw_bf16, per_token, bias, acc_out, y, M, N, K, row_inv};
    static_assert(!kFused || FM == 1, "the fused form takes up to 16 tokens");
    constexpr int RED = kWaves * FM * 256 * 4;  // partial sums: [wave][16 FM tokens][16 columns]
    __shared__ __attribute__((aligned(16))) unsigned char lds[kFused && kFusedLds > RED ? kFusedLds : RED];
    __shared__ float sx_lds[16];
    __shared__ unsigned red_key[kWaves];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, h = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const int units = K / 128;
    const int xs = K + 16;  // kFused: bytes per token row in LDS (the 16 spread the rows over the banks)

    // ---- activations first: loads return in order
    u32x4_t xv[PT];
    const u32x4_t *xp = reinterpret_cast<const u32x4_t *>(p.xf);
    const int pieces = kFused ? p.M * (K / 8) : 0;
    if constexpr (kFused) {
        if (!p.per_token) {
#pragma unroll
            for (int t = 0; t < PT; ++t) {
                const int i = tid + t * kThreads;
                xv[t] = xp[i < pieces ? i : 0];
            }
        }
    }

    const unsigned char *wrow = p.w + (long long)(n0 + r) * K + 16 * h;
    u32x4_t wv[UB][2], xf[UB][FM][2];
    auto load_units = [&](int u0) {
#pragma unroll
        for (int b = 0; b < UB; ++b) {
            const int u = u0 + b * kWaves;
            const int uc = u < units ? u : 0;  // past the end: any line, its product is skipped
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                wv[b][t] = *reinterpret_cast<const u32x4_t *>(wrow + uc * 128 + 64 * t);
                if constexpr (!kFused) {
#pragma unroll
                    for (int j = 0; j < FM; ++j) {
                        const int m = 16 * j + r;
                        xf[b][j][t] = *reinterpret_cast<const u32x4_t *>(p.x8 + (long long)(m < p.M ? m : p.M - 1) * K + uc * 128 + 64 * t + 16 * h);
                    }
                }
            }
        }
    };
    load_units(wave);

    if constexpr (kFused) {
        const int row16 = K / 8;  // pieces per token
        auto put = [&](int i, u32x2_t q) {
            const int m = (int)__umulhi((unsigned)i, p.row_inv);  // i / row16 (i and row16 below 2^14)
            *reinterpret_cast<u32x2_t *>(lds + m * xs + (i - m * row16) * 8) = q;
        };
        if (p.per_token) {
            // a wave per token row
            for (int m = wave; m < p.M; m += kWaves) {
                const u32x4_t *row = xp + (long long)m * row16;
                // The row in steps of four pieces a lane, requested together (past the end: the lane's first again), the first
                // step's kept for the second pass. Left to the compiler's unrolling, each load waited for the use of the one before:
                // 2304 x 9216 at 4 tokens 16.4 us -> 13.8, 1280 x 5120 at 12 14.7 -> 12.0. Many rows of a short K leave no
                // registers for it beside a second workgroup on the unit (10240 x 2560 at 16 tokens 22.9, one at a time 20.1).
                constexpr int STEP = PT == 16 && UB == 2 ? 1 : 4;
                constexpr bool KEEP = STEP == 4;
                auto load = [&](u32x4_t (&v)[STEP], int i) {
#pragma unroll
                    for (int t = 0; t < STEP; ++t) v[t] = row[i + 64 * t < row16 ? i + 64 * t : lane < row16 ? lane : 0];
                };
                u32x4_t head[STEP];
                if constexpr (KEEP) load(head, lane);
                auto in_steps = [&](auto use) {
                    if constexpr (KEEP)
#pragma unroll
                        for (int t = 0; t < STEP; ++t) use(lane + 64 * t, head[t]);
                    for (int i = KEEP ? lane + 64 * STEP : lane; i < row16; i += 64 * STEP) {
                        u32x4_t v[STEP];
                        load(v, i);
#pragma unroll
                        for (int t = 0; t < STEP; ++t) use(i + 64 * t, v[t]);
                    }
                };
                act_u16x2_t most = {0, 0};
                in_steps([&](int, const u32x4_t &v) { most = act_amax8(v, most); });
                const unsigned amax = wave_max_u32(act_amax_of(most));
                const float am = __uint_as_float(amax << 16);
                const float inv = am == 0.0f ? 0.0f : 127.0f / am;
                if (lane == 0) sx_lds[m] = am / 127.0f;
                auto quantise = [&](auto finite) {
                    in_steps([&](int i, const u32x4_t &v) {
                        if (i < row16) put(m * row16 + i, act_quant8_token(v, inv, decltype(finite)::value));
                    });
                };
                if (act_finite_row(am, inv)) quantise(std::true_type());
                else quantise(std::false_type());
            }
        } else {
            MaxKeys keys;
#pragma unroll
            for (int t = 0; t < PT; ++t)
                if (tid + t * kThreads < pieces) keys.add8(xv[t]);
            unsigned k = wave_max_u32(keys.key());
            if (lane == 0) red_key[wave] = k;
            __syncthreads();
#pragma unroll
            for (int w = 0; w < kWaves; ++w) k = k > red_key[w] ? k : red_key[w];
            const float c = max_key_value(k);
            if (tid < 16) sx_lds[tid] = c * (1.0f / 127.0f);
#pragma unroll
            for (int t = 0; t < PT; ++t)
                if (tid + t * kThreads < pieces) put(tid + t * kThreads, act_quant8_any<true>(xv[t], c));
        }
        __syncthreads();
    }

    i32x4_t acc[FM];
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[j] = i32x4_t{0, 0, 0, 0};
    const unsigned char *xrow = lds + (r < p.M ? r : p.M - 1) * xs + 16 * h;
    for (int u0 = wave; u0 < units; u0 += UB * kWaves) {
        u32x4_t wc[UB][2], xc[UB][FM][2];
#pragma unroll
        for (int b = 0; b < UB; ++b)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                wc[b][t] = wv[b][t];
#pragma unroll
                for (int j = 0; j < FM; ++j) xc[b][j][t] = xf[b][j][t];
            }
        if (u0 + UB * kWaves < units) load_units(u0 + UB * kWaves);
#pragma unroll
        for (int b = 0; b < UB; ++b) {
            const int u = u0 + b * kWaves;
            if (u >= units) break;
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < FM; ++j) {
                    u32x4_t x;
                    if constexpr (kFused) x = *reinterpret_cast<const u32x4_t *>(xrow + u * 128 + 64 * t);
                    else x = xc[b][j][t];
                    acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, wc[b][t]), __builtin_bit_cast(i32x4_t, x), acc[j], 0, 0, 0);
                }
        }
    }

    // ---- the eight partial sums (the activations in LDS have been read)
    if constexpr (kFused) __syncthreads();
    int *part = reinterpret_cast<int *>(lds);
#pragma unroll
    for (int j = 0; j < FM; ++j) *reinterpret_cast<i32x4_t *>(part + ((wave * FM + j) * 16 + r) * 16 + 4 * h) = acc[j];
    __syncthreads();
    for (int i = tid; i < FM * 256; i += kThreads) {
        const int m = i >> 4, n = n0 + (i & 15);
        if (m >= p.M) continue;
        int s = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) s += part[w * FM * 256 + i];
        const float sw = p.sw_bf16 ? lq_bf16_bits_to_f32(reinterpret_cast<const unsigned short *>(p.sw)[n]) : reinterpret_cast<const float *>(p.sw)[n];
        float v = ((float)s * (kFused ? sx_lds[m] : p.sx[m])) * sw;
        if (p.bias) v += lq_bf16_bits_to_f32(p.bias[n]);
        p.y[(long long)m * p.N + n] = lq_f32_to_bf16_bits(v);
        if (p.acc_out) p.acc_out[(long long)m * p.N + n] = s;
    }
}

}  // namespace

template <class Kernel>
static void launch_gemv8(Kernel kernel, const Gemv8Params &p, const void *x, hipStream_t st) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.N / 16)), dim3(kThreads), 0, st, x, p.w, p.M, p.N, p.K, p.row_inv, p.per_token, p.sw_bf16, p.sw,
                       p.bias, p.y, p.sx, p.acc_out);
}

// Called by lq_a8w8_fwd (lq_gemm.hip) after argument validation: K % 128 == 0, N % 16 == 0, M <= 32.
int lq_gemv_i8_launch(const void *x8, const void *w8, const float *sx, const void *sw, bool sw_bf16, const void *bias, void *y,
                      int *acc_or_null, int M, int N, int K, hipStream_t st) {
    Gemv8Params p = {};
    p.x8 = (const unsigned char *)x8; p.w = (const unsigned char *)w8; p.sx = sx; p.sw = sw; p.sw_bf16 = sw_bf16;
    p.bias = (const unsigned short *)bias; p.y = (unsigned short *)y; p.acc_out = acc_or_null;
    p.M = M; p.N = N; p.K = K;
    if (M > 16) launch_gemv8(gemv_i8_kernel<2, false, 2>, p, p.x8, st);
    else if (K >= kDeep) launch_gemv8(gemv_i8_kernel<1, false, 4>, p, p.x8, st);
    else launch_gemv8(gemv_i8_kernel<1, false, 2>, p, p.x8, st);
    return lq_check_launch("lq_a8w8_fwd");
}

template <int PT>
static void launch_fused(const Gemv8Params &p, hipStream_t st) {
    if (p.K >= kDeep) launch_gemv8(gemv_i8_kernel<1, true, 4, PT>, p, p.xf, st);
    else launch_gemv8(gemv_i8_kernel<1, true, 2, PT>, p, p.xf, st);
}

extern "C" int lq_a8w8_infer_takes(int64_t M, int64_t N, int64_t K) {
    return M >= 1 && M <= 16 && N >= 16 && N % 16 == 0 && N < (1ll << 31) && K >= 128 && K % 128 == 0 && M * (K + 16) <= kFusedLds;
}

extern "C" int lq_a8w8_infer(const void *x, const void *w, const void *qscales_bf16, const void *bias_or_null, void *y, int per_token,
                             int64_t M, int64_t N, int64_t K, void *stream) {
    LQ_REQUIRE(x && w && qscales_bf16 && y, "lq_a8w8_infer: null pointer argument");
    LQ_REQUIRE(lq_a8w8_infer_takes(M, N, K), "lq_a8w8_infer: M=%lld N=%lld K=%lld: see lq_a8w8_infer_takes", (long long)M, (long long)N, (long long)K);
    LQ_REQUIRE(lq_aligned(x, 16) && lq_aligned(w, 16) && lq_aligned(y, 16) && lq_aligned(qscales_bf16, 2),
               "lq_a8w8_infer: x, w and y must be 16-byte aligned");
    Gemv8Params p = {};
    p.xf = (const unsigned short *)x; p.w = (const unsigned char *)w; p.sw = qscales_bf16; p.sw_bf16 = 1; p.per_token = per_token != 0;
    p.bias = (const unsigned short *)bias_or_null; p.y = (unsigned short *)y;
    p.M = (int)M; p.N = (int)N; p.K = (int)K;
    p.row_inv = (unsigned)(((1ull << 32) + (unsigned long long)(K / 8) - 1) / (unsigned long long)(K / 8));
    const long long pieces = M * (K / 8);
    hipStream_t st = (hipStream_t)stream;
    if (pieces <= 4 * kThreads) launch_fused<4>(p, st);
    else if (pieces <= 8 * kThreads) launch_fused<8>(p, st);
    else launch_fused<16>(p, st);  // 64 KB of int8 are 8192 pieces
    return lq_check_launch("lq_a8w8_infer");
}
