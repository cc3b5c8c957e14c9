// Everything a block-layout GEMM reads, prepared in one launch: x_hat of one tensor (optionally LayerNorm first) in the
// 32-row block layout, and the fp16 weights of up to two layers reconstructed from their packed codes.
//
// Latency-bound up to a few thousand rows (it is one dependent chain: load -> LayerNorm sums -> group sums -> codes ->
// store, beside another: codes -> lookups -> store), vector-ALU-bound beyond.  What the split of the work does about it:
//   * A wave owns whole rows when there is a LayerNorm (two lanes per group, 2 G lanes per row, as many rows as fit 64
//     lanes), so the row sums stay inside the wave: no workgroup barrier, and the number of workgroups is rows / 8 (G =
//     16) instead of rows / 32.  (act_quant_rows_ln_kernel owns 32 rows per workgroup and meets at five barriers: 18 us
//     at 591 x 1024 where this takes 7.)  Without one a wave owns 8 or more rows x up to four groups.
//   * x_hat goes to the block layout through LDS in runs of at least 8 rows x 16 bytes, i.e. whole 128-byte lines
//     wherever the tensor's rows allow it.
//   * Weights: a wave owns 32 output columns x four groups, lane = (column, half group): 32 codes, one set of metadata
//     and four 16-byte stores per group and lane, every store of the wave two 512-byte runs of the weight block layout.
//     All index arithmetic is 32-bit.  (weight_dequant8_kernel owns 8 weights per thread: the 64-bit division and the
//     three metadata loads per 8 weights made it 10 us for 4096 x 1024; here 4.)
// FP8 operands (F8): the same work with pieces of 16 values and rows padded with zeros to 128 values.
// Arithmetic: arcq_act_quant_core.h and the stage-2 expression, unchanged -- bit-identical to the stand-alone kernels.
#include "arcq_act_quant_core.h"
#include "arcq_gemm.h"

namespace arcq {
namespace {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kPrepWaves = 4;
constexpr int kPrepThreads = 64 * kPrepWaves;

struct PrepWeights {
    const uint8_t *packed;
    const float *cb, *center, *scale, *code_sum;
    void *out;               // [N/32][K/8][32][8] fp16, or [N][K] if row_major; FP8: [N/32][Kp/16][32][16] or [N][Kp]
    int N, G;                // G = K / 64
    float mult;              // FP8: power of two in front of the rounding
    int row_major;
    unsigned blocks;         // workgroups (0: no such job)
};

template <int BITS>
__device__ __forceinline__ void prep_load_codes(const uint8_t *__restrict__ p, uint32_t (&w)[BITS])
{
    if constexpr (BITS == 4) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t *>(p);
        w[0] = v[0]; w[1] = v[1]; w[2] = v[2]; w[3] = v[3];
    } else if constexpr (BITS == 2) {
        const u32x2_t v = *reinterpret_cast<const u32x2_t *>(p);
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

// One wave: columns 32 nb ... + 31 of groups 4 gq ... + 3 of a layer's weights.  `lut`: the codebook per lane.
template <int BITS, bool F8>
__device__ __forceinline__ void prep_weights(const PrepWeights &w, unsigned block, float *lut)
{
    constexpr int L = 1 << BITS;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int quads = (w.G + 3) >> 2;
    const int item = static_cast<int>(block) * kPrepWaves + wave;
    const int nb = item / quads, g0 = (item - nb * quads) * 4;
    const bool mine = nb * 32 < w.N;
    const int n = nb * 32 + (lane & 31), half = lane >> 5;
    const int ng = mine ? min(4, w.G - g0) : 0;
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
    if (threadIdx.x < 64) {
#pragma unroll
        for (int q = 0; q < L; ++q) lut[q * 64 + lane] = w.cb[q];
    }
    __syncthreads();
    const char *lut_lane = reinterpret_cast<const char *>(lut) + lane * 4;
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
        for (int e = 0; e < 32; ++e) v[e] = *reinterpret_cast<const float *>(lut_lane + (prep_code_at<BITS>(codes[i], e) << 8));
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
    const int lane = threadIdx.x & 63;
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
    if (threadIdx.x < 64) {
#pragma unroll
        for (int q = 0; q < L; ++q) lut[q * 64 + lane] = w.cb[q];
    }
    __syncthreads();
    if (!mine) return;
    uint32_t o[4] = {0, 0, 0, 0};
    if constexpr (F8) {
        if (!padding) {
            float v[32];
#pragma unroll
            for (int e = 0; e < 16; ++e) v[e] = lut[(((e < 8 ? codes : more) >> (BITS * (e & 7))) & (L - 1)) * 64 + lane];
            weights_fp8x16(v, 0, m, s, c, w.mult, o);
        }
        store_writethrough16(static_cast<char *>(w.out) + static_cast<int64_t>(idx) * 16, o[0], o[1], o[2], o[3]);
        return;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        float v[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) v[e] = fma_f32(lut[((codes >> (BITS * (2 * d + e))) & (L - 1)) * 64 + lane] - m, s, c);
        const __half2 h = __floats2half2_rn(v[0], v[1]);
        o[d] = *reinterpret_cast<const uint32_t *>(&h);
    }
    store_writethrough16(static_cast<char *>(w.out) + static_cast<int64_t>(idx) * 16, o[0], o[1], o[2], o[3]);
}

// F8 (LN = false only): FP8 operands.
// LN = true: LayerNorm over the rows first; GC = all G groups of a row (2 GC lanes per row).
// LN = false: a wave takes R rows x GC groups; consecutive waves take consecutive group chunks.
// rows_per_wave = R; chunks = group chunks per row (1 with a LayerNorm).
template <typename TIN, int BITS, bool LN, bool F8>
__global__ void __launch_bounds__(kPrepThreads)
prepare_kernel(const TIN *__restrict__ x, const float *__restrict__ gamma, const float *__restrict__ beta, float ln_eps,
               const float *__restrict__ thr, const float *__restrict__ cb, char *__restrict__ x_hat, float eps, int rows,
               int G, int GC, int R, int chunks, int tiles, PrepWeights w0, PrepWeights w1)
{
    constexpr int L = 1 << BITS;
    constexpr int kIn = 32 * static_cast<int>(sizeof(TIN)) / 16;       // 16-byte loads per lane (32 values)
    extern __shared__ __attribute__((aligned(16))) unsigned char prep_smem[];
    __shared__ float lut[L * 64];
    __shared__ Bucket table[kMaxBuckets + 1];
    __shared__ int slow_slots[kPrepWaves];
    // The weight workgroups come first: they are the longer chain where the rows are few.
    if (blockIdx.x < w0.blocks + w1.blocks) {
        const bool second = blockIdx.x >= w0.blocks;
        const PrepWeights &w = second ? w1 : w0;
        const unsigned block = blockIdx.x - (second ? w0.blocks : 0);
        if (w.row_major) prep_weights_rows<BITS, F8>(w, block, lut);
        else prep_weights<BITS, F8>(w, block, lut);
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wg = blockIdx.x - (w0.blocks + w1.blocks), wgs = gridDim.x - (w0.blocks + w1.blocks);
    const int P = 2 * GC;                                   // lanes per row
    const int rl = lane / P, pl = lane - rl * P;            // row of the wave, lane of the row
    const int K = G * 64;
    const bool lane_used = rl < R;
    unsigned char *tile = prep_smem;                         // LN: the workgroup's; else wave-private
    float *part = reinterpret_cast<float *>(prep_smem + (LN ? kPrepWaves * R * GC * 128 : kPrepWaves * 4096)) + wave * (64 + 16);
    const int pstride = P;                                   // partial sums of a row

    // Tile t: rows t0 ... of chunk ch.  With a LayerNorm a tile is the workgroup's 4 R rows (wave w rows R w ...);
    // without one it is a wave's R rows x GC groups, numbered chunk-fastest.
    uint4 raw[kIn];
    int row, g0;
    bool valid;
    auto locate = [&](int t) {
        if constexpr (LN) {
            row = t * (kPrepWaves * R) + wave * R + rl;
            g0 = 0;
            valid = lane_used && t < tiles && row < rows;
        } else {
            const int rt = t / chunks;
            row = rt * R + rl;
            g0 = (t - rt * chunks) * GC;
            valid = lane_used && t < tiles && row < rows && g0 + (pl >> 1) < G;
        }
    };
    auto fetch = [&](int t) {
        locate(t);
        const uint4 *p = reinterpret_cast<const uint4 *>(x + static_cast<int64_t>(valid ? row : 0) * K + (valid ? g0 * 64 + pl * 32 : 0));
#pragma unroll
        for (int i = 0; i < kIn; ++i) raw[i] = valid ? p[i] : make_uint4(0, 0, 0, 0);
    };
    const int first = LN ? wg : wg * kPrepWaves + wave;
    const int step = LN ? wgs : wgs * kPrepWaves;
    fetch(first);
    float th[L - 1], cbv[L];
    load_quant_params<BITS>(thr, cb, th, cbv);
    const BucketScale bq = pick_bucket_scale<BITS>(th);
    build_quant_tables_by<BITS>(th, cbv, bq, lut, table, slow_slots, tid, kPrepThreads);      // while the first tile is on its way
    __syncthreads();
    bool table_ok = true;
#pragma unroll
    for (int w = 0; w < kPrepWaves; ++w) table_ok = table_ok && (slow_slots[w] == 0);
    const float fk = static_cast<float>(K);
    constexpr int kPieces = F8 ? 4 : 8;                     // 16-byte pieces of a group of x_hat
    const int row_groups = F8 ? (G + 1) / 2 * 2 : G;        // with the padding
    const int row_bytes = row_groups * kPieces * 16;

    const int trips = (tiles + (LN ? 1 : kPrepWaves) * wgs - 1) / ((LN ? 1 : kPrepWaves) * wgs);      // the same for every wave
    for (int trip = 0, t = first; trip < trips; ++trip, t += step) {
        float xv[32];
        if constexpr (sizeof(TIN) == 2) {
#pragma unroll
            for (int i = 0; i < kIn; ++i) {
                const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    xv[i * 8 + 2 * d] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] & 0xffffu)));
                    xv[i * 8 + 2 * d + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] >> 16)));
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < kIn; ++i) {
                xv[4 * i] = __uint_as_float(raw[i].x); xv[4 * i + 1] = __uint_as_float(raw[i].y);
                xv[4 * i + 2] = __uint_as_float(raw[i].z); xv[4 * i + 3] = __uint_as_float(raw[i].w);
            }
        }
        const int my_row = row, my_g0 = g0;
        const bool my_valid = valid;
        if (trip + 1 < trips) fetch(t + step);            // the next tile loads under this one's arithmetic
        if constexpr (LN) {
            // Row sums: every lane folds its 32 values serially, the row's 2 G partial sums are added in a fixed order
            // (group by group, lower half first) by every lane of the row.  The partial sums go through wave-private
            // LDS, whose operations execute in order.
            auto row_total = [&](float mine) {
                if (lane_used) part[rl * pstride + pl] = mine;
                __builtin_amdgcn_wave_barrier();
                const float *src = part + (lane_used ? rl : 0) * pstride;
                float acc = 0.0f;
                for (int i = 0; i < P; i += 2) {
                    const float2 v = *reinterpret_cast<const float2 *>(src + i);
                    acc += v.x;
                    acc += v.y;
                }
                __builtin_amdgcn_wave_barrier();
                return acc;
            };
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) a += xv[j];
            const float mean = row_total(a) / fk;
            float q = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                xv[j] -= mean;
                const float sq = xv[j] * xv[j];
                q += sq;
            }
            const float rstd = 1.0f / sqrtf(row_total(q) / fk + ln_eps);
            const float4 *gp = reinterpret_cast<const float4 *>(gamma + (lane_used ? pl : 0) * 32);
            const float4 *bp = reinterpret_cast<const float4 *>(beta + (lane_used ? pl : 0) * 32);
#pragma unroll
            for (int j4 = 0; j4 < 8; ++j4) {
                const float4 gv = gp[j4], bv = bp[j4];
                const float g4[4] = {gv.x, gv.y, gv.z, gv.w}, b4[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float tv = xv[4 * j4 + e] * rstd;
                    const float u = tv * g4[e];
                    float yv = u + b4[e];
                    if constexpr (sizeof(TIN) == 2) yv = __half2float(__float2half_rn(yv));     // what a LayerNorm kernel stores
                    xv[4 * j4 + e] = yv;
                }
            }
        }
        float mu, var, s, sum_codes;
        group_stats32x2(xv, eps, mu, var, s);
        group_codes32x2<BITS>(xv, mu, var, s, th, bq, table, lut, table_ok, lane, sum_codes);
        const float code_mean = sum_codes * 0.015625f;
        uint4 o[kPieces / 2];
#pragma unroll
        for (int i = 0; i < kPieces / 2; ++i) {
            uint32_t w[4];
            if constexpr (F8) {
                xhat_fp8x16(xv, 16 * i, s, code_mean, mu, w);
            } else {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const int j = 8 * i + 2 * d;
                    const __half2 h = __floats2half2_rn(fma_f32(s, xv[j] - code_mean, mu), fma_f32(s, xv[j + 1] - code_mean, mu));
                    w[d] = *reinterpret_cast<const uint32_t *>(&h);
                }
            }
            o[i] = make_uint4(w[0], w[1], w[2], w[3]);
        }
        // ---- out: piece (k, row) at LDS slot k * rows_in_tile + row, then 16 bytes per lane, rows fastest ----
        if constexpr (LN) {
            const int RW = kPrepWaves * R;
            if (lane_used) {
#pragma unroll
                for (int i = 0; i < kPieces / 2; ++i)
                    *reinterpret_cast<uint4 *>(tile + ((pl * (kPieces / 2) + i) * RW + wave * R + rl) * 16) = o[i];
            }
            __syncthreads();
            const int r0 = t * RW;
            const int pieces = GC * kPieces * RW;
            for (int p = tid; p < pieces; p += kPrepThreads) {
                const int k = p / RW, r = p - k * RW;
                const int rr = r0 + r;
                if (rr < rows) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(tile + p * 16);
                    const int blk = rr >> 5, nrows = min(32, rows - blk * 32);
                    store_writethrough16(x_hat + static_cast<int64_t>(blk) * 32 * row_bytes + (k * nrows + (rr & 31)) * 16, v.x, v.y, v.z, v.w);
                }
            }
            __syncthreads();
        } else {
            unsigned char *mine = tile + wave * 4096;
            if (lane_used) {
#pragma unroll
                for (int i = 0; i < kPieces / 2; ++i) *reinterpret_cast<uint4 *>(mine + ((pl * (kPieces / 2) + i) * R + rl) * 16) = o[i];
            }
            __builtin_amdgcn_wave_barrier();
            // R is a power of two and R * GC = 32 here: 256 pieces, four per lane (FP8: two)
            const int rt0 = my_row - rl;
#pragma unroll
            for (int i = 0; i < kPieces / 2; ++i) {
                const int p = i * 64 + lane;
                const int k = p / R, r = p - k * R;
                const int rr = rt0 + r;
                if (rr < rows && t < tiles && my_g0 * kPieces + k < G * kPieces) {
                    const uint4 v = *reinterpret_cast<const uint4 *>(mine + p * 16);
                    const int blk = rr >> 5, nrows = min(32, rows - blk * 32);
                    char *dst = x_hat + static_cast<int64_t>(blk) * 32 * row_bytes + ((my_g0 * kPieces + k) * nrows + (rr & 31)) * 16;
                    store_writethrough16(dst, v.x, v.y, v.z, v.w);
                    // (an odd number of groups: GC = 1, and the last group's tile writes the padding group too)
                    if (F8 && row_groups > G && my_g0 == G - 1) store_writethrough16(dst + kPieces * nrows * 16, 0, 0, 0, 0);
                }
            }
            __builtin_amdgcn_wave_barrier();
            (void)my_valid;
        }
    }
}

template <typename TIN, bool F8>
void launch_prepare_t(const arcq_prepare_args &a, const PrepWeights &w0, const PrepWeights &w1, hipStream_t stream)
{
    const int G = static_cast<int>(a.K / 64), rows = static_cast<int>(a.rows);
    const bool ln = a.ln_weight != nullptr;
    int GC, R, chunks, tiles, wgs;
    size_t smem;
    if (ln) {
        GC = G;
        R = 64 / (2 * G);
        chunks = 1;
        tiles = (rows + kPrepWaves * R - 1) / (kPrepWaves * R);
        wgs = tiles;
        smem = static_cast<size_t>(kPrepWaves) * R * GC * 128;
    } else {
        GC = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1;
        R = 32 / GC;
        chunks = G / GC;
        tiles = ((rows + R - 1) / R) * chunks;
        wgs = (tiles + kPrepWaves - 1) / kPrepWaves;
        smem = kPrepWaves * 4096;
    }
    smem += kPrepWaves * (64 + 16) * sizeof(float);
    // Beyond four workgroups per CU the waves walk their tiles: the lookup tables are built once per workgroup.
    const int cap = 4 * device_cus();
    if (rows == 0) wgs = 0;
    else if (wgs > cap) wgs = cap;
    const unsigned grid = w0.blocks + w1.blocks + static_cast<unsigned>(wgs);
    if (grid == 0) return;
#define ARCQ_LAUNCH_PREP(B, LNV)                                                                                              \
    do {                                                                                                                       \
        hipLaunchKernelGGL((prepare_kernel<TIN, B, LNV, F8>), dim3(grid), dim3(kPrepThreads), smem, stream,                    \
                           static_cast<const TIN *>(a.x), a.ln_weight, a.ln_bias, a.ln_eps, a.thresholds, a.codebook,          \
                           static_cast<char *>(a.x_hat), 1.0e-6f, rows, G, GC, R, chunks, tiles, w0, w1);                      \
    } while (0)
    if constexpr (!F8) {
        if (ln) {
            if (a.bits == 4) ARCQ_LAUNCH_PREP(4, true);
            else if (a.bits == 3) ARCQ_LAUNCH_PREP(3, true);
            else ARCQ_LAUNCH_PREP(2, true);
            return;
        }
    }
    if (a.bits == 4) ARCQ_LAUNCH_PREP(4, false);
    else if (a.bits == 3) ARCQ_LAUNCH_PREP(3, false);
    else ARCQ_LAUNCH_PREP(2, false);
#undef ARCQ_LAUNCH_PREP
}

}  // namespace
}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_prepare(const arcq_prepare_args *a, void *stream)
{
    if (!a) return fail(ARCQ_ERR_NULL, "arcq_prepare: args must not be NULL");
    if (!bits_ok(a->bits)) return fail(ARCQ_ERR_BITS, "arcq_prepare: bits must be 2, 3, or 4");
    if (a->rows < 0 || a->K < 0) return fail(ARCQ_ERR_SHAPE, "arcq_prepare: bad sizes");
    PrepWeights pw[2] = {};
    for (int i = 0; i < 2; ++i) {
        const arcq_prepare_weights &w = a->weights[i];
        if (!w.packed) continue;
        if (w.N <= 0 || w.K <= 0 || (!w.row_major && w.N % 32 != 0) || w.K % 64 != 0)
            return fail(ARCQ_ERR_SHAPE, "arcq_prepare: weights need N a multiple of 32 (column blocks) and K a multiple of 64 (got %lld x %lld)",
                        static_cast<long long>(w.N), static_cast<long long>(w.K));
        if (w.N * w.K >= (int64_t(1) << 31)) return fail(ARCQ_ERR_SHAPE, "arcq_prepare: weight tensor too large");
        if (!w.codebook || !w.center || !w.scale || !w.code_sum || !w.w_hat) return fail(ARCQ_ERR_NULL, "arcq_prepare: NULL weight tensor pointer");
        if (!aligned(w.w_hat, 16) || !aligned(w.packed, 16)) return fail(ARCQ_ERR_ALIGN, "arcq_prepare: w_hat and packed must be 16-byte aligned");
        const int G = static_cast<int>(w.K / 64);
        // workgroups: waves of 32 columns x 4 groups, or threads of a piece
        if (a->fp8 && !(w.w_mult > 0.0f)) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_prepare: w_mult must be positive");
        const int row_pieces = a->fp8 ? (G + 1) / 2 * 8 : G * 8;
        const unsigned items = w.row_major ? static_cast<unsigned>((w.N * row_pieces + 63) / 64) : static_cast<unsigned>(w.N / 32) * ((G + 3) / 4);
        pw[i] = PrepWeights{w.packed, w.codebook, w.center, w.scale, w.code_sum, w.w_hat, static_cast<int>(w.N), G, w.w_mult,
                            w.row_major != 0, (items + kPrepWaves - 1) / kPrepWaves};
    }
    if (a->rows > 0) {
        if (a->K % 64 != 0 || a->K == 0) return fail(ARCQ_ERR_GROUP, "arcq_prepare: in_features must be a positive multiple of 64");
        if (a->x_dtype != ARCQ_F16 && a->x_dtype != ARCQ_F32) return fail(ARCQ_ERR_DTYPE, "arcq_prepare: x must be float16 or float32");
        if (!a->x || !a->thresholds || !a->codebook || !a->x_hat) return fail(ARCQ_ERR_NULL, "arcq_prepare: NULL tensor pointer");
        if (a->x == a->x_hat) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_prepare: x_hat must not alias x");
        if (a->rows >= (int64_t(1) << 26) || a->rows * a->K >= (int64_t(1) << 31)) return fail(ARCQ_ERR_SHAPE, "arcq_prepare: tensor too large");
        if (a->ln_weight && (!a->ln_bias || a->K > 2048 || a->fp8))
            return fail(ARCQ_ERR_UNSUPPORTED, "arcq_prepare: the LayerNorm needs weight and bias, in_features <= 2048 and fp16 operands");
        if (!aligned(a->x, 16) || !aligned(a->x_hat, 16) || !aligned(a->ln_weight, 16) || !aligned(a->ln_bias, 16))
            return fail(ARCQ_ERR_ALIGN, "arcq_prepare: x, x_hat, ln_weight and ln_bias must be 16-byte aligned");
    }
    if (a->rows == 0 && !pw[0].blocks && !pw[1].blocks) return ARCQ_OK;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->fp8) {
        if (a->x_dtype == ARCQ_F32) launch_prepare_t<float, true>(*a, pw[0], pw[1], st);
        else launch_prepare_t<__half, true>(*a, pw[0], pw[1], st);
    } else if (a->x_dtype == ARCQ_F32) {
        launch_prepare_t<float, false>(*a, pw[0], pw[1], st);
    } else {
        launch_prepare_t<__half, false>(*a, pw[0], pw[1], st);
    }
    return launch_status("arcq_prepare");
}
