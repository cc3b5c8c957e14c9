// Weights of a layer reconstructed by extra workgroups in front of a stage-1 launch's grid.
//
// A wave owns 32 output columns x four groups (fewer in small layers), lane = (column, half group): 32 codes, one set of metadata
// and four 16-byte stores per group and lane, every store of the wave two 512-byte runs of the weight block layout.
// All index arithmetic is 32-bit.  (weight_dequant8_kernel owns 8 weights per thread: the 64-bit division and the
// three metadata loads per 8 weights made it 10 us for 4096 x 1024; here 4.)
#pragma once

#include "arcq_act_quant_core.h"

namespace arcq {

typedef uint32_t u32x4_prep_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_prep_t __attribute__((ext_vector_type(2)));

constexpr int kPrepWaves = 4;
constexpr int kPrepThreads = 64 * kPrepWaves;

struct PrepWeights {
    const uint8_t *packed;
    const float *cb, *center, *scale, *code_sum;
    void *out;               // [N/32][K/8][32][8] fp16, or [N][K] if row_major; FP8: [N/32][Kp/16][32][16] or [N][Kp]
    int N, G;                // G = K / 64
    float mult;              // FP8: power of two in front of the rounding
    int row_major;
    int wave_groups;         // column blocks: groups per wave (1, 2 or 4)
    unsigned blocks;         // workgroups (0: no such job)
};

template <int BITS>
__device__ __forceinline__ void prep_load_codes(const uint8_t *__restrict__ p, uint32_t (&w)[BITS])
{
    if constexpr (BITS == 4) {
        const u32x4_prep_t v = *reinterpret_cast<const u32x4_prep_t *>(p);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
    } else if constexpr (BITS == 2) {
        const u32x2_prep_t v = *reinterpret_cast<const u32x2_prep_t *>(p);
        w[0] = v[0]; w[1] = v[1];
    } else {
        const uint32_t *q = reinterpret_cast<const uint32_t *>(p);
        w[0] = q[0]; w[1] = q[1]; w[2] = q[2];
    }
}
template <int BITS>
__device__ __forceinline__ uint32_t prep_code_at(const uint32_t (&w)[BITS], int q)
{
    const int bit = q * BITS;
    const int d = bit >> 5, sh = bit & 31;
    uint32_t v = w[d] >> sh;
    if (sh + BITS > 32) v |= w[d + 1] << (32 - sh);
    return v & ((1u << BITS) - 1u);
}

// Sixteen reconstructed weights times `mult` as one FP8 piece.
__device__ __forceinline__ void weights_fp8x16(const float (&v)[32], int j0, float mg, float s, float c, float mult, uint32_t (&o)[4])
{
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = fma_f32(v[j0 + 8 * p + e] - mg, s, c) * mult;
        to_fp8x8(t, o[2 * p], o[2 * p + 1]);
    }
}

// One wave: columns 32 nb ... + 31 of `wave_groups` groups of a layer's weights.  `lut`: LDS for the codebook.
template <int BITS, bool F8>
__device__ __forceinline__ void prep_weights(const PrepWeights &w, unsigned block, float *lut)
{
    constexpr int L = 1 << BITS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int runs = (w.G + w.wave_groups - 1) / w.wave_groups;
    const int item = static_cast<int>(block) * kPrepWaves + wave;
    const int nb = item / runs, g0 = (item - nb * runs) * w.wave_groups;
    const bool mine = nb * 32 < w.N;
    const int n = nb * 32 + (lane & 31), half = lane >> 5;
    const int ng = mine ? min(w.wave_groups, w.G - g0) : 0;
    uint32_t codes[4][BITS];
    float c[4], s[4], m[4];
    const uint8_t *src = w.packed + static_cast<int64_t>(n) * (w.G * 8 * BITS) + g0 * (8 * BITS) + half * (4 * BITS);
    const int64_t mi = static_cast<int64_t>(n) * w.G + g0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < ng) {
            prep_load_codes<BITS>(src + i * 8 * BITS, codes[i]);
            c[i] = w.center[mi + i];
            s[i] = w.scale[mi + i];
            m[i] = w.code_sum[mi + i];
        }
    if (threadIdx.x < L) lut[threadIdx.x] = w.cb[threadIdx.x];
    __syncthreads();
    const int row_groups = F8 ? (w.G + 1) / 2 * 2 : w.G;
    constexpr int kPieces = F8 ? 4 : 8;            // 16-byte pieces of a group
    char *dst = static_cast<char *>(w.out) + static_cast<int64_t>(nb) * (row_groups * kPieces * 512) + (g0 * kPieces + half * (kPieces / 2)) * 512 +
                (lane & 31) * 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= ng) break;
        const float mg = m[i] * 0.015625f;          // S/64, exact
        float v[32];
#pragma unroll
        for (int e = 0; e < 32; ++e) v[e] = lut[prep_code_at<BITS>(codes[i], e)];
#pragma unroll
        for (int p = 0; p < kPieces / 2; ++p) {
            uint32_t o[4];
            if constexpr (F8) {
                weights_fp8x16(v, 16 * p, mg, s[i], c[i], w.mult, o);
            } else {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const __half2 h = __floats2half2_rn(fma_f32(v[p * 8 + 2 * d] - mg, s[i], c[i]), fma_f32(v[p * 8 + 2 * d + 1] - mg, s[i], c[i]));
                    o[d] = *reinterpret_cast<const uint32_t *>(&h);
                }
            }
            store_writethrough16(dst + (i * kPieces + p) * 512, o[0], o[1], o[2], o[3]);
        }
    }
    if (F8 && mine && g0 + ng == w.G && row_groups > w.G) {
#pragma unroll
        for (int p = 0; p < 2; ++p) store_writethrough16(dst + (ng * kPieces + p) * 512, 0, 0, 0, 0);
    }
}

// Row-major output: a 16-byte piece per thread, consecutive threads consecutive pieces of a row.
template <int BITS, bool F8>
__device__ __forceinline__ void prep_weights_rows(const PrepWeights &w, unsigned block, float *lut)
{
    constexpr int L = 1 << BITS;
    constexpr uint32_t kPieces = F8 ? 4 : 8;       // of a group
    const uint32_t live = static_cast<uint32_t>(w.G) * kPieces;
    const uint32_t per_row = F8 ? (live + 7) / 8 * 8 : live;
    const uint32_t idx = block * kPrepThreads + threadIdx.x;
    const bool mine = idx < static_cast<uint32_t>(w.N) * per_row;
    const uint32_t n = mine ? idx / per_row : 0, at = mine ? idx - n * per_row : 0;
    const bool padding = at >= live;
    const uint32_t k = padding ? 0 : at;
    const uint8_t *src = w.packed + static_cast<int64_t>(n * live + k) * ((F8 ? 2 : 1) * BITS);
    const uint32_t codes = load_codes8<BITS>(src), more = F8 ? load_codes8<BITS>(src + BITS) : 0;
    const int64_t mi = static_cast<int64_t>(n) * w.G + k / kPieces;
    const float c = w.center[mi], s = w.scale[mi], m = w.code_sum[mi] * 0.015625f;
    if (threadIdx.x < L) lut[threadIdx.x] = w.cb[threadIdx.x];
    __syncthreads();
    if (!mine) return;
    uint32_t o[4] = {0, 0, 0, 0};
    if constexpr (F8) {
        if (!padding) {
            float v[32];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = lut[((e < 8 ? codes : more) >> (BITS * (e & 7))) & (L - 1)];
            weights_fp8x16(v, 0, m, s, c, w.mult, o);
        }
        store_writethrough16(static_cast<char *>(w.out) + static_cast<int64_t>(idx) * 16, o[0], o[1], o[2], o[3]);
        return;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) v[e] = fma_f32(lut[(codes >> (BITS * (2 * d + e))) & (L - 1)] - m, s, c);
        const __half2 h = __floats2half2_rn(v[0], v[1]);
        o[d] = *reinterpret_cast<const uint32_t *>(&h);
    }
    store_writethrough16(static_cast<char *>(w.out) + static_cast<int64_t>(idx) * 16, o[0], o[1], o[2], o[3]);
}

// Weight workgroups come first: they are the longer chain where the rows are few.
template <int BITS, bool F8>
__device__ __forceinline__ bool prep_weight_workgroup(const PrepWeights &w0, const PrepWeights &w1, float *lut)
{
    if (blockIdx.x >= w0.blocks + w1.blocks) return false;
    if (threadIdx.x >= kPrepThreads) {          // a table builder has nothing to do here; the job's one barrier counts it
        __syncthreads();
        return true;
    }
    const bool second = blockIdx.x >= w0.blocks;
    const PrepWeights &w = second ? w1 : w0;
    const unsigned block = blockIdx.x - (second ? w0.blocks : 0);
    if (w.row_major) prep_weights_rows<BITS, F8>(w, block, lut);
    else prep_weights<BITS, F8>(w, block, lut);
    return true;
}

inline PrepWeights weight_job(const arcq_prepare_weights &w, bool fp8)
{
    const int G = static_cast<int>(w.K / 64);
    const int row_pieces = fp8 ? (G + 1) / 2 * 8 : G * 8;
    // Groups per wave: four while that makes two waves for every SIMD; a smaller job is as long as one wave's chain, and a wave
    // with one group is done a microsecond or two earlier.
    const unsigned columns = static_cast<unsigned>(w.N / 32);
    const int wg = columns * G >= 8192u ? 4 : columns * G >= 4096u ? 2 : 1;
    // workgroups: waves of 32 columns x wg groups, or threads of a piece
    const unsigned items = w.row_major ? static_cast<unsigned>((w.N * row_pieces + 63) / 64) : columns * ((G + wg - 1) / wg);
    return PrepWeights{w.packed, w.codebook, w.center, w.scale, w.code_sum, w.w_hat, static_cast<int>(w.N), G, w.w_mult,
                       w.row_major != 0, wg, (items + kPrepWaves - 1) / kPrepWaves};
}

// The job of a caller's description (packed == NULL: none), checked.
inline int weight_job_checked(const char *fn, const arcq_prepare_weights *w, bool fp8, PrepWeights &out)
{
    out = PrepWeights{};
    if (!w || !w->packed) return ARCQ_OK;
    if (w->N <= 0 || w->K <= 0 || (!w->row_major && w->N % 32 != 0) || w->K % 64 != 0)
        return fail(ARCQ_ERR_SHAPE, "%s: weights need N a multiple of 32 (column blocks) and K a multiple of 64 (got %lld x %lld)", fn,
                    static_cast<long long>(w->N), static_cast<long long>(w->K));
    if (w->N * w->K >= (int64_t(1) << 31)) return fail(ARCQ_ERR_SHAPE, "%s: weight tensor too large", fn);
    if (!w->codebook || !w->center || !w->scale || !w->code_sum || !w->w_hat) return fail(ARCQ_ERR_NULL, "%s: NULL weight tensor pointer", fn);
    if (!aligned(w->w_hat, 16) || !aligned(w->packed, 16)) return fail(ARCQ_ERR_ALIGN, "%s: w_hat and packed must be 16-byte aligned", fn);
    if (fp8 && !(w->w_mult > 0.0f)) return fail(ARCQ_ERR_UNSUPPORTED, "%s: w_mult must be positive", fn);
    out = weight_job(*w, fp8);
    return ARCQ_OK;
}

}  // namespace arcq
