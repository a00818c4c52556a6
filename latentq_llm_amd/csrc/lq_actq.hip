// Activation quantisers in front of the int8 GEMM (bf16 -> int8 + the per-row scales its epilogue reads):
//   lq_act_quant_i8           per-tensor, clamp value given (a device scalar)
//   lq_act_quant_i8_dynamic   per-tensor, clamp value = the tensor's own maximum (one or two launches, no host sync)
//   lq_act_quant_i8_per_token one scale per token row from the row's absolute maximum (one pass over HBM)
// and, for the backward passes, lq_act_dequant_i8 (int8 -> bf16) and lq_act_fake_quant (bf16 -> bf16 on the int8 grid)
#include "lq_common.h"
#include "lq_actq_math.h"

namespace {

// The 8 elements from `base` on, for the clamp value c (uniform over the launch; kOwnMax: x's maximum).
template <bool kOwnMax>
__device__ __forceinline__ void act_quant_piece(const unsigned short *__restrict__ x, signed char *__restrict__ x8, long long base,
                                                long long n, float c) {
    if (base >= n) return;
    if (base + 8 <= n && (((uintptr_t)(x + base)) & 15) == 0 && (((uintptr_t)(x8 + base)) & 7) == 0) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(x + base);
        *reinterpret_cast<u32x2_t *>(x8 + base) = act_quant8_any<kOwnMax>(v, c);
    } else {
        for (long long i = base; i < n && i < base + 8; ++i) {
            float f = lq_bf16_bits_to_f32(x[i]);
            float a = lq_bf16r(f * 127.0f);
            float q = lq_bf16r(a / c);
            float rr = q == q ? __builtin_amdgcn_fmed3f(rintf(q), -128.0f, 127.0f) : 0.0f;
            x8[i] = (signed char)(int)rr;
        }
    }
}

__global__ __launch_bounds__(256) void act_quant_kernel(const unsigned short *__restrict__ x,
                                                        const float *__restrict__ clampv, signed char *__restrict__ x8,
                                                        long long n) {
    act_quant_piece<false>(x, x8, ((long long)blockIdx.x * 256 + threadIdx.x) * 8, n, clampv[0]);
}

// ---- the tensor's own maximum as clamp value ---------------------------------------------------
// Maximum over a workgroup of 256 threads, returned to every thread.
__device__ __forceinline__ unsigned wg_max_u32(unsigned v, unsigned *red) {
    v = wave_max_u32(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const unsigned a = red[0] > red[1] ? red[0] : red[1], b = red[2] > red[3] ? red[2] : red[3];
    return a > b ? a : b;
}

constexpr int kMaxPartials = LQ_ACT_WORK_FLOATS - 8;

// Phase 1: workgroup b writes the largest key of its grid-stride share of x to partial[b].
__global__ __launch_bounds__(256) void tensor_max_kernel(const unsigned short *__restrict__ x, long long n,
                                                         unsigned *__restrict__ partial) {
    __shared__ unsigned red[4];
    MaxKeys keys;
    const long long n8 = n / 8;
    const u32x4_t *x16 = reinterpret_cast<const u32x4_t *>(x);
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n8; i += (long long)gridDim.x * 256) {
        const u32x4_t v = x16[i];
        keys.add8(v);
    }
    unsigned k = keys.key();
    if (blockIdx.x == 0 && (long long)threadIdx.x < n - n8 * 8) {
        const unsigned t = max_key(x[n8 * 8 + threadIdx.x]);
        k = k > t ? k : t;
    }
    k = wg_max_u32(k, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = k;
}

// what follows once the largest key is known: the clamp value and alpha to `work`, the per-row scales, and the thread's 8 elements
__device__ __forceinline__ void act_quant_with_key(unsigned k, const unsigned short *__restrict__ x, signed char *__restrict__ x8,
                                                   float *__restrict__ sx, float *__restrict__ work, long long n, long long M, int alpha_bf16) {
    const float c = max_key_value(k);
    float alpha = c * (1.0f / 127.0f);
    if (alpha_bf16) alpha = lq_bf16r(alpha);
    const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid == 0) {
        work[0] = c;
        work[1] = alpha;
    }
    for (long long m = gid; m < M; m += (long long)gridDim.x * blockDim.x) sx[m] = alpha;
    act_quant_piece<true>(x, x8, gid * 8, n, c);
}

// Both phases in one launch, for few elements: every workgroup finds the maximum of all of them. An int8 layer with two launches
// and with one, us: 17 x 2048 9.0 / 8.8, 32 x 2048 9.5 / 9.5, 59 x 2048 12.1 / 14.2, 95 x 2048 12.3 / 16.0. A launch is 3 us of
// the host's time besides, which such calls wait for.
constexpr long long kOneLaunch = 80 << 10;
__global__ __launch_bounds__(1024) void act_quant_one_kernel(const unsigned short *__restrict__ x, signed char *__restrict__ x8,
                                                             float *__restrict__ sx, float *__restrict__ work, int n, int M, int alpha_bf16) {
    __shared__ __attribute__((aligned(16))) unsigned red[16];
    MaxKeys keys;
    const int n8 = n / 8;
    const u32x4_t *x16 = reinterpret_cast<const u32x4_t *>(x);
#pragma unroll 8
    for (int i = threadIdx.x; i < n8; i += 1024) keys.add8(x16[i]);
    unsigned k = keys.key();
    if ((int)threadIdx.x < n - n8 * 8) {
        const unsigned t = max_key(x[n8 * 8 + threadIdx.x]);
        k = k > t ? k : t;
    }
    k = wave_max_u32(k);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = k;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 16; w += 4) {
        const u32x4_t r = *reinterpret_cast<const u32x4_t *>(red + w);
#pragma unroll
        for (int j = 0; j < 4; ++j) k = k > r[j] ? k : r[j];
    }
    act_quant_with_key(k, x, x8, sx, work, n, M, alpha_bf16);
}

// Phase 2: every workgroup reduces the partial keys to the clamp value, then quantises its 2048 elements;
// the first M threads of the grid also write the per-row scale alpha = clampv * fl(1/127) (the tensor library
// divides a tensor by a host scalar as a product with the scalar's fp32 reciprocal), rounded to bf16 when the
// caller's alpha is a bf16 tensor.
__global__ __launch_bounds__(256) void act_quant_dyn_kernel(const unsigned short *__restrict__ x, signed char *__restrict__ x8,
                                                            float *__restrict__ sx, float *__restrict__ work, int partials,
                                                            long long n, long long M, int alpha_bf16) {
    __shared__ unsigned red[4];
    const unsigned *partial = reinterpret_cast<const unsigned *>(work + 8);
    unsigned k = 0u;
    for (int i = threadIdx.x; i < partials; i += 256) k = k > partial[i] ? k : partial[i];
    k = wg_max_u32(k, red);
    act_quant_with_key(k, x, x8, sx, work, n, M, alpha_bf16);
}

// ---- one scale per token row --------------------------------------------------------------------
// A wave owns a row: the row's largest |x| (as a bit pattern: magnitudes order like unsigned integers, and a NaN
// pattern is above infinity, so a NaN in the row ends up in the scale), then
//   sx[m] = amax / 127,   x8 = clamp(rint(x * (127 / amax)), -128, 127)      (fp32, IEEE division, NaN -> 0)
// with 127 / amax replaced by 0 for an all-zero row. A lane keeps PT 16-byte pieces of the row in registers between
// the two phases (rows of up to 512 * PT elements are read from memory once); longer rows are read again.
template <int PT>
__global__ __launch_bounds__(256) void act_quant_token_kernel(const unsigned short *__restrict__ x, signed char *__restrict__ x8,
                                                              float *__restrict__ sx, int M, int K) {
    const int lane = threadIdx.x & 63;
    const int m = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
    if (m >= M) return;
    const u32x4_t *row = reinterpret_cast<const u32x4_t *>(x + (long long)m * K);
    u32x2_t *out = reinterpret_cast<u32x2_t *>(x8 + (long long)m * K);
    const int n16 = K / 8, T = (n16 + 63) / 64;
    u32x4_t v[PT];
    act_u16x2_t most = {0, 0};
    auto take = [&](const u32x4_t &w) { most = act_amax8(w, most); };
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int i = lane + 64 * t;
        v[t] = u32x4_t{0u, 0u, 0u, 0u};
        if (i < n16) v[t] = row[i];
    }
#pragma unroll
    for (int t = 0; t < PT; ++t) take(v[t]);
    for (int t = PT; t < T; ++t) {
        const int i = lane + 64 * t;
        if (i < n16) take(row[i]);
    }
    const unsigned amax = wave_max_u32(act_amax_of(most));
    const float am = __uint_as_float(amax << 16);
    const float inv = am == 0.0f ? 0.0f : 127.0f / am;
    if (lane == 0) sx[m] = am / 127.0f;
    const bool finite = act_finite_row(am, inv);
    auto quant = [&](const u32x4_t &w) { return act_quant8_token(w, inv, finite); };
#pragma unroll
    for (int t = 0; t < PT; ++t) {
        const int i = lane + 64 * t;
        if (i < n16) out[i] = quant(v[t]);
    }
    for (int t = PT; t < T; ++t) {
        const int i = lane + 64 * t;
        if (i < n16) out[i] = quant(row[i]);
    }
}

// The way back, for the backward pass: out = bf16(x8 * bf16(s)) with s = scale[m] (per token) or scale[0]; the values of
// `x8.to(dtype) * s.to(dtype)`. 16 elements per thread (one row: K % 16 == 0).
__global__ __launch_bounds__(256) void act_dequant_kernel(const u32x4_t *__restrict__ x8, const float *__restrict__ scale,
                                                          u32x4_t *__restrict__ out, long long n_chunks, long long chunks_per_row,
                                                          int per_token) {
    const long long L = (long long)blockIdx.x * 256 + threadIdx.x;
    if (L >= n_chunks) return;
    const float s = lq_bf16r(scale[per_token ? L / chunks_per_row : 0]);
    const u32x4_t c = x8[L];
    u32x4_t o[2];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float v[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) v[b] = (float)(int)(signed char)((c[w] >> (8 * b)) & 0xFFu) * s;
        o[w >> 1][2 * (w & 1)] = lq_pack_bf16(v[0], v[1]);
        o[w >> 1][2 * (w & 1) + 1] = lq_pack_bf16(v[2], v[3]);
    }
    out[2 * L] = o[0];
    out[2 * L + 1] = o[1];
}

// Fake quantisation for the backward pass of the layers that keep the bf16 activations (utils/quant.py:200-202,
// 358-360): out = bf16(clamp(rne(bf16(x * s)), -128, 127) / s) with the bf16 scalar s = 127 / clampv, i.e. the chain
// (input * s).round_().clamp_(-128, 127).div_(s) as one pass; 8 elements per thread. The quotient of an integer of at
// most 8 bits and a bf16 number keeps 2^-17 (relative) from every bf16 rounding tie, so for 2^-40 <= |s| <= 2^40 the
// product with RN(1 / s) rounds to the same bf16 number as the quotient; other scales take the division. NaN stays NaN.
__global__ __launch_bounds__(256) void act_fake_quant_kernel(const unsigned short *__restrict__ x, const unsigned short *__restrict__ s_dev,
                                                             unsigned short *__restrict__ out, long long n) {
    const float s = lq_bf16_bits_to_f32(s_dev[0]);
    const bool fast = fabsf(s) >= 0x1p-40f && fabsf(s) <= 0x1p40f;
    const float r = 1.0f / s;
    const long long base = ((long long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (base >= n) return;
    auto one = [&](float f) {
        const float a = lq_bf16r(f * s);
        const float q = a != a ? a : __builtin_amdgcn_fmed3f(rintf(a), -128.0f, 127.0f);
        return fast ? q * r : q / s;
    };
    if (base + 8 <= n) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(x + base);
        u32x4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = lq_pack_bf16(one(lq_bf16_lo(v[j])), one(lq_bf16_hi(v[j])));
        *reinterpret_cast<u32x4_t *>(out + base) = o;
    } else {
        for (long long i = base; i < n; ++i) out[i] = lq_f32_to_bf16_bits(one(lq_bf16_bits_to_f32(x[i])));
    }
}

}  // namespace

extern "C" int lq_act_fake_quant(const void *x, const void *s_bf16_dev, void *out, int64_t n, void *stream) {
    LQ_REQUIRE(x && s_bf16_dev && out && n >= 0, "lq_act_fake_quant: bad argument");
    LQ_REQUIRE(lq_aligned(x, 16) && lq_aligned(out, 16) && lq_aligned(s_bf16_dev, 2),
               "lq_act_fake_quant: x and out must be 16-byte aligned");
    if (n == 0) return LQ_OK;
    const long long blocks = ((n + 7) / 8 + 255) / 256;
    LQ_REQUIRE(blocks <= 0x7FFFFFFFll, "lq_act_fake_quant: n too large");
    hipLaunchKernelGGL(act_fake_quant_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)x,
                       (const unsigned short *)s_bf16_dev, (unsigned short *)out, (long long)n);
    return lq_check_launch("lq_act_fake_quant");
}

extern "C" int lq_act_dequant_i8(const int8_t *x8, const float *scale, int per_token, void *out, int64_t M, int64_t K,
                                 void *stream) {
    LQ_REQUIRE(x8 && scale && out, "lq_act_dequant_i8: null pointer argument");
    LQ_REQUIRE(M > 0 && K > 0 && K % 16 == 0 && M < (1ll << 31) && K < (1ll << 31),
               "lq_act_dequant_i8: need M > 0 and K a positive multiple of 16 (M=%lld K=%lld)", (long long)M, (long long)K);
    LQ_REQUIRE(lq_aligned(x8, 16) && lq_aligned(out, 16) && lq_aligned(scale, 4),
               "lq_act_dequant_i8: x8 and out must be 16-byte aligned, scale 4-byte");
    const long long n_chunks = M * K / 16;
    const long long blocks = (n_chunks + 255) / 256;
    LQ_REQUIRE(blocks <= 0x7FFFFFFFll, "lq_act_dequant_i8: tensor too large");
    hipLaunchKernelGGL(act_dequant_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const u32x4_t *)x8, scale,
                       (u32x4_t *)out, n_chunks, (long long)(K / 16), per_token);
    return lq_check_launch("lq_act_dequant_i8");
}

extern "C" int lq_act_quant_i8(const void *x, const float *clampv_dev, int8_t *x8, int64_t n, void *stream) {
    LQ_REQUIRE(x && clampv_dev && x8 && n >= 0, "lq_act_quant_i8: bad argument");
    if (n == 0) return LQ_OK;
    const long long blocks = ((n + 7) / 8 + 255) / 256;
    LQ_REQUIRE(blocks <= 0x7FFFFFFFll, "lq_act_quant_i8: n too large");
    hipLaunchKernelGGL(act_quant_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const unsigned short *)x, clampv_dev, (signed char *)x8, (long long)n);
    return lq_check_launch("lq_act_quant_i8");
}

extern "C" int lq_act_quant_i8_dynamic(const void *x, int8_t *x8, float *sx, float *work, int64_t M, int64_t K, int alpha_bf16,
                                       void *stream) {
    LQ_REQUIRE(x && x8 && sx && work, "lq_act_quant_i8_dynamic: null pointer argument");
    LQ_REQUIRE(M > 0 && K > 0 && M < (1ll << 31) && K < (1ll << 31), "lq_act_quant_i8_dynamic: M=%lld and K=%lld must be positive",
               (long long)M, (long long)K);
    LQ_REQUIRE(lq_aligned(x, 16) && lq_aligned(x8, 8) && lq_aligned(sx, 4) && lq_aligned(work, 4),
               "lq_act_quant_i8_dynamic: x must be 16-byte aligned, x8 8-byte, sx and work 4-byte");
    const long long n = M * K;
    const long long blocks = ((n + 7) / 8 + 255) / 256;
    LQ_REQUIRE(blocks <= 0x7FFFFFFFll, "lq_act_quant_i8_dynamic: tensor too large");
    if (n <= kOneLaunch) {
        hipLaunchKernelGGL(act_quant_one_kernel, dim3((unsigned)((n + 8191) / 8192)), dim3(1024), 0, (hipStream_t)stream,
                           (const unsigned short *)x, (signed char *)x8, sx, work, (int)n, (int)M, alpha_bf16);
        return lq_check_launch("lq_act_quant_i8_dynamic");
    }
    const int partials = (int)(blocks < kMaxPartials ? blocks : kMaxPartials);
    hipLaunchKernelGGL(tensor_max_kernel, dim3((unsigned)partials), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)x, n,
                       reinterpret_cast<unsigned *>(work + 8));
    int rc = lq_check_launch("lq_act_quant_i8_dynamic(max)");
    if (rc) return rc;
    hipLaunchKernelGGL(act_quant_dyn_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)x,
                       (signed char *)x8, sx, work, partials, n, (long long)M, alpha_bf16);
    return lq_check_launch("lq_act_quant_i8_dynamic");
}

extern "C" int lq_act_quant_i8_per_token(const void *x, int8_t *x8, float *sx, int64_t M, int64_t K, void *stream) {
    LQ_REQUIRE(x && x8 && sx, "lq_act_quant_i8_per_token: null pointer argument");
    LQ_REQUIRE(M > 0 && K > 0 && K % 8 == 0 && M < (1ll << 31) && K < (1ll << 31),
               "lq_act_quant_i8_per_token: need M > 0 and K a positive multiple of 8 (M=%lld K=%lld)", (long long)M, (long long)K);
    LQ_REQUIRE(lq_aligned(x, 16) && lq_aligned(x8, 8) && lq_aligned(sx, 4),
               "lq_act_quant_i8_per_token: x must be 16-byte aligned, x8 8-byte, sx 4-byte");
    const unsigned blocks = (unsigned)((M + 3) / 4);
    if (K <= 2048)
        hipLaunchKernelGGL(act_quant_token_kernel<4>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)x,
                           (signed char *)x8, sx, (int)M, (int)K);
    else
        hipLaunchKernelGGL(act_quant_token_kernel<16>, dim3(blocks), dim3(256), 0, (hipStream_t)stream, (const unsigned short *)x,
                           (signed char *)x8, sx, (int)M, (int)K);
    return lq_check_launch("lq_act_quant_i8_per_token");
}
