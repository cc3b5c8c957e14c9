// Stage 1 of a quantized patch-embedding convolution (QuantConv2dPCARCQ with kernel == stride, FQ/quant_backends.py:
// 329-384): every pixel's three channels are one quantization group (its act_group_size is min(64, in_channels) = 3),
// and the reconstructed values are written straight as the rows of the patch matrix the convolution multiplies,
// row = patch (b, py, px), column k = c * 256 + i * 16 + j -- row-major [M, 768] fp16, or in the 32-row block layout
// [M/32][96][32][8] that arcq_linear_fused_blocked reads (a last block of r < 32 rows as [96][r][8]).
//
// The arithmetic per group is that of the any-group-size kernel of arcq_act_quant (which restates
// EXT/arcq_activation_kernel.cu:24-77 for a group of three): serial sums from zero, mean and variance divided by the
// group size with IEEE divisions, t = d / s, compare chain, x_hat = fma(s, cb[code] - code_sum / 3, mu) -- so the values
// equal, bit for bit, what that kernel writes for the NHWC pixels; what is new is the order of the work: one wave = 32
// patches x one pixel row of theirs, a lane = eight neighbouring pixels, loads and stores of 16 contiguous bytes, no
// NHWC copy of the image and no gather of the patch rows afterwards.
//
// Bound by the vector ALUs.  With plain divisions (six of them a pixel, about ten instructions each) and the compare chain (45
// instructions a value at four bits) a pixel took 230 instructions and 64 images 28 us, 19 MB in and 19 MB out (8 us at the copy
// rate).  The means are therefore products with fused corrections, the codes bucket lookups without a quotient as in
// arcq_act_quant_core.h, and root and reciprocal come from one hardware reciprocal root: about 85 instructions a pixel, 128 images
// 16.1 us and 256 32.2 (IEEE's square root and division expanded by the compiler, quotients by fused corrections and every wave
// building the tables: 256 42.4).  Waves walk their items so that a workgroup builds its tables once.
#include "arcq_prepare_core.h"
#include "arcq_gemm.h"

#include <algorithm>

namespace arcq {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kP = 16, kC = 3, kKP = kC * kP * kP;      // patch side, channels, 768 values per patch row

// v / 3 rounded to nearest: the product with RN(1/3), which is within a unit in the last place, and one fused correction.  Exact
// while the residual stays in the normal range (every mantissa checked on the CPU; |v| >= 2^-100 or v = 0).
__device__ __forceinline__ float third_of(float v)
{
    const float q = v * (1.0f / 3.0f);
    return __fmaf_rn(__fmaf_rn(-3.0f, q, v), 1.0f / 3.0f, q);
}
// The square root rounded to nearest, from the hardware's reciprocal root by one coupled iteration (Goldschmidt) and a fused
// correction: equal to sqrtf for every float of [2^-100, 2^100) from any reciprocal root within one unit in the last place, which is the
// instruction's accuracy (every mantissa of an even and an odd binade checked on the CPU), at a third of sqrtf's instructions.  y: the
// reciprocal, within 2^-22.
__device__ __forceinline__ float sqrt_and_reciprocal(float a, float &y)
{
    const float r = __builtin_amdgcn_rsqf(a);
    float g = a * r, h = 0.5f * r;
    const float e = __fmaf_rn(-h, g, 0.5f);
    g = __fmaf_rn(g, e, g);
    h = __fmaf_rn(h, e, h);
    y = h + h;
    return __fmaf_rn(__fmaf_rn(-g, g, a), h, g);
}
__device__ __forceinline__ bool in_range(float v) { return (v == 0.0f) | ((fabsf(v) >= 0x1p-60f) & (fabsf(v) <= 0x1p60f)); }

// The fast form looks every value up before it is known to be in range (what it finds otherwise is not used): the payload of an
// fp32 NaN may name any of the offsets that code_offset_of can form (that of an fp16 one, widened, has no bits there): its table has
// all those entries.  And the sign of a NaN remainder may make one code more than there are, which reads the member behind `cb`.
template <typename TIN> constexpr int kTableEntries = sizeof(TIN) == 4 ? 0x1ff8 / static_cast<int>(sizeof(Bucket)) + 1 : kMaxBuckets + 1;

// Eight pixels quantized and reconstructed in place, every operation rounded as IEEE has it.
template <int BITS, typename Tables>
__device__ __forceinline__ void quantize_pixels(float (&x)[8][kC], float eps, const Tables &q)
{
    constexpr float fgs = static_cast<float>(kC);
    float mu[8], s[8];
    uint32_t at[8][kC];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float sum = 0.0f, var = 0.0f;
#pragma unroll
        for (int c = 0; c < kC; ++c) sum += x[e][c];
        mu[e] = sum / fgs;
#pragma unroll
        for (int c = 0; c < kC; ++c) {
            x[e][c] -= mu[e];
            var += x[e][c] * x[e][c];
        }
        s[e] = sqrtf(var / fgs + eps);
#pragma unroll
        for (int c = 0; c < kC; ++c) x[e][c] = x[e][c] / s[e];
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) bisect_codes<BITS>(x[e], q.thr, at[e]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float sum_codes = 0.0f;
#pragma unroll
        for (int c = 0; c < kC; ++c) {
            x[e][c] = code_value(q.cb, at[e][c]);
            sum_codes += x[e][c];
        }
        const float code_mean = sum_codes / fgs;
#pragma unroll
        for (int c = 0; c < kC; ++c) x[e][c] = fma_f32(s[e], x[e][c] - code_mean, mu[e]);
    }
}

// One pixel on the tables.  Returns whether every intermediate was in the range where the result is the above's.  SIMPLE (fp16
// input, eps >= 2^-30, codebook values 0 or within 2^+-60): the sums are multiples of 2^-24 or of 2^-83 and cannot be too small,
// a variance below 2^-60 vanishes beside eps, d_c is 0 or a multiple of 2^-49, and whatever is not finite shows in s.
template <int BITS, bool SIMPLE, typename Tables>
__device__ __forceinline__ bool quantize_pixel_fast(float (&x)[kC], float eps, const BucketScale &bq, const Tables &q)
{
    float sum = 0.0f;
#pragma unroll
    for (int c = 0; c < kC; ++c) sum += x[c];
    const float mu = third_of(sum);
    float var = 0.0f;
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        x[c] -= mu;
        var += x[c] * x[c];
    }
    float y;
    const float s = sqrt_and_reciprocal(third_of(var) + eps, y);
    const CodeScale cs = code_scale_of(s, y, bq);
    float sum_codes = 0.0f;
#pragma unroll
    for (int c = 0; c < kC; ++c) {
        const float v = code_value(q.cb, code_offset_of(x[c], cs, bq, q.bucket));
        x[c] = v;
        sum_codes += v;
    }
    const float code_mean = third_of(sum_codes);
#pragma unroll
    for (int c = 0; c < kC; ++c) x[c] = fma_f32(s, x[c] - code_mean, mu);
    const bool root_ok = (s >= 0x1p-50f) & (s < 0x1p50f);
    if constexpr (SIMPLE) return root_ok;
    // d_c is 0 or at least 2^-90 once |mu| >= 2^-66 or all of them are 0.
    // (No short circuits: a branch per pixel would keep the eight pixels of a lane from overlapping.)
    const bool means_ok = !((fabsf(mu) < 0x1p-66f) & (var > 0.0f));
    return in_range(sum) & in_range(var) & in_range(sum_codes) & root_ok & means_ok;
}

template <typename TIN, int BITS>
__global__ void __launch_bounds__(kPrepThreads)
act_quant_patches_kernel(const TIN *__restrict__ img, const float *__restrict__ thr, const float *__restrict__ cb,
                         __half *__restrict__ x_hat, int B, int H, int W, float eps, int blocked, int items, PrepWeights weights)
{
    constexpr int L = 1 << BITS;
    constexpr int kIn = 8 * static_cast<int>(sizeof(TIN)) / 16;
    __shared__ QuantTablesOf<kTableEntries<TIN>> tables;
    if (prep_weight_workgroup<BITS, false>(weights, PrepWeights{}, tables.cb)) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int lr = lane & 31, lh = lane >> 5;
    const int pw = W / kP, np = (H / kP) * pw;
    const int M = B * np;
    const int64_t plane = static_cast<int64_t>(H) * W;
    const int step = (gridDim.x - weights.blocks) * kPrepWaves;
    int item = (blockIdx.x - weights.blocks) * kPrepWaves + (tid >> 6);      // (block of 32 patches, pixel row i)
    uint4 raw[kC][kIn];
    auto fetch = [&](int it) {
        it = min(it, items - 1);
        const int m = min((it >> 4) * 32 + lr, M - 1), i = it & 15;
        const int b = m / np, p = m - b * np, py = p / pw, px = p - py * pw;
        const TIN *src = img + (static_cast<int64_t>(b) * kC * H + py * kP + i) * W + px * kP + 8 * lh;
#pragma unroll
        for (int c = 0; c < kC; ++c)
#pragma unroll
            for (int j = 0; j < kIn; ++j) raw[c][j] = reinterpret_cast<const uint4 *>(src + c * plane)[j];
    };
    QuantParams params{};
    if (tid < 64) params = load_quant_params<BITS>(thr, cb, lane);
    fetch(item);
    if (tid < 64) {
        build_quant_tables<BITS>(params, tables, lane);
        if constexpr (sizeof(TIN) == 4)
            for (int b = tables.geometry.nb + 1 + lane; b < kTableEntries<TIN>; b += 64) tables.bucket[b] = Bucket{__builtin_huge_valf(), 0};
    }
    __syncthreads();
    constexpr bool kSimple = sizeof(TIN) == 2;
    const BucketScale bq = tables.geometry;
    const bool table_ok = tables.usable && (!kSimple || (eps >= 0x1p-30f && __all(in_range(tables.cb[lane & (L - 1)]))));

    for (; item < items; item += step) {
        float x[8][kC];
        auto unpack = [&]() {
#pragma unroll
            for (int c = 0; c < kC; ++c)
#pragma unroll
                for (int j = 0; j < kIn; ++j) {
                    const uint32_t w[4] = {raw[c][j].x, raw[c][j].y, raw[c][j].z, raw[c][j].w};
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        if constexpr (sizeof(TIN) == 2) {
                            x[2 * d][c] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] & 0xffffu)));
                            x[2 * d + 1][c] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] >> 16)));
                        } else {
                            x[4 * j + d][c] = __uint_as_float(w[d]);
                        }
                    }
                }
        };
        unpack();
        bool ok = table_ok;
#pragma unroll
        for (int e = 0; e < 8; ++e) ok = ok & quantize_pixel_fast<BITS, kSimple>(x[e], eps, bq, tables);
        if (!__all(ok)) {
            unpack();
            quantize_pixels<BITS>(x, eps, tables);
        }
        const int blk = item >> 4, i = item & 15, m = blk * 32 + lr;
        fetch(item + step);                                    // (the next item's pixels while this one's leave)
        if (m < M) {
            // piece column of (c, i, half): k / 8 = c * 32 + 2 i + lh
            const int rows = min(32, M - blk * 32);
#pragma unroll
            for (int c = 0; c < kC; ++c) {
                const int kp = c * 32 + 2 * i + lh;
                __half *dst = blocked ? x_hat + static_cast<int64_t>(blk) * 32 * kKP + (static_cast<int64_t>(kp) * rows + lr) * 8
                                      : x_hat + static_cast<int64_t>(m) * kKP + kp * 8;
                uint32_t o[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const __half2 h = __floats2half2_rn(x[2 * d][c], x[2 * d + 1][c]);
                    o[d] = *reinterpret_cast<const uint32_t *>(&h);
                }
                store_writethrough16(dst, o[0], o[1], o[2], o[3]);
            }
        }
    }
}

template <typename TIN, int BITS>
void launch_patches(const void *img, const float *thr, const float *cb, void *x_hat, int B, int H, int W, float eps, int blocked,
                    const PrepWeights &weights, hipStream_t stream)
{
    const int64_t M = static_cast<int64_t>(B) * (H / kP) * (W / kP);
    const int items = static_cast<int>((M + 31) / 32 * 16);
    // (what the chip holds at once: 256 images 35.7 us against 38.3 with four workgroups per CU and 39.3 with six, all before the
    // codes were found without a quotient)
    const int wgs = std::min((items + kPrepWaves - 1) / kPrepWaves, 5 * device_cus());
    hipLaunchKernelGGL((act_quant_patches_kernel<TIN, BITS>), dim3(weights.blocks + wgs), dim3(kPrepThreads), 0, stream,
                       static_cast<const TIN *>(img), thr, cb, static_cast<__half *>(x_hat), B, H, W, eps, blocked, items, weights);
}

int patches_checked(const char *fn, const void *img, int img_dtype, const float *thresholds, const float *codebook, void *x_hat, int64_t B,
                    int64_t C, int64_t H, int64_t W, int64_t patch, int bits, float eps, int blocked, const PrepWeights &weights,
                    void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "%s: bits must be 2, 3, or 4", fn);
    if (B < 0 || H < 0 || W < 0) return fail(ARCQ_ERR_SHAPE, "%s: negative size", fn);
    if (C != kC || patch != kP)
        return fail(ARCQ_ERR_UNSUPPORTED, "%s: three channels and 16 x 16 patches only (got C=%lld, patch=%lld)", fn,
                    static_cast<long long>(C), static_cast<long long>(patch));
    if (H % kP || W % kP) return fail(ARCQ_ERR_SHAPE, "%s: image sides must be multiples of 16", fn);
    if (img_dtype != ARCQ_F32 && img_dtype != ARCQ_F16) return fail(ARCQ_ERR_DTYPE, "%s: img must be float32 or float16", fn);
    if (B * H * W == 0) return ARCQ_OK;
    if (!img || !thresholds || !codebook || !x_hat) return fail(ARCQ_ERR_NULL, "%s: NULL pointer", fn);
    if (!aligned(img, 16) || !aligned(x_hat, 16)) return fail(ARCQ_ERR_ALIGN, "%s: img and x_hat must be 16-byte aligned", fn);
    if (B > (1 << 20) || H > (1 << 14) || W > (1 << 14) || B * (H / kP) * (W / kP) >= (int64_t(1) << 26))
        return fail(ARCQ_ERR_SHAPE, "%s: tensor too large", fn);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int b = static_cast<int>(B), h = static_cast<int>(H), w = static_cast<int>(W);
#define ARCQ_GO(T) \
    do { \
        if (bits == 4) launch_patches<T, 4>(img, thresholds, codebook, x_hat, b, h, w, eps, blocked, weights, st); \
        else if (bits == 3) launch_patches<T, 3>(img, thresholds, codebook, x_hat, b, h, w, eps, blocked, weights, st); \
        else launch_patches<T, 2>(img, thresholds, codebook, x_hat, b, h, w, eps, blocked, weights, st); \
    } while (0)
    if (img_dtype == ARCQ_F16) ARCQ_GO(__half);
    else ARCQ_GO(float);
#undef ARCQ_GO
    return launch_status(fn);
}

}  // namespace
}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_act_quant_patches(const void *img, int img_dtype, const float *thresholds, const float *codebook, void *x_hat,
                                    int64_t B, int64_t C, int64_t H, int64_t W, int64_t patch, int bits, float eps, int blocked,
                                    void *stream)
{
    return patches_checked("arcq_act_quant_patches", img, img_dtype, thresholds, codebook, x_hat, B, C, H, W, patch, bits, eps, blocked,
                           PrepWeights{}, stream);
}

ARCQ_API int arcq_prepare_patches(const void *img, int img_dtype, const float *thresholds, const float *codebook, void *x_hat, int64_t B,
                                  int64_t C, int64_t H, int64_t W, int64_t patch, int bits, float eps, const arcq_prepare_weights *weights,
                                  void *stream)
{
    PrepWeights w;
    const int rc = weight_job_checked("arcq_prepare_patches", weights, false, w);
    if (rc != ARCQ_OK) return rc;
    return patches_checked("arcq_prepare_patches", img, img_dtype, thresholds, codebook, x_hat, B, C, H, W, patch, bits, eps, 1, w, stream);
}
