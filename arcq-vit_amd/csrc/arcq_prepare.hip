// Everything a block-layout GEMM reads, prepared in one launch: x_hat of one tensor (optionally LayerNorm first) in the
// 32-row block layout, and the fp16 weights of up to two layers reconstructed from their packed codes.
//
// Latency-bound up to a few thousand rows (it is one dependent chain: load -> LayerNorm sums -> group sums -> codes ->
// store, beside another: codes -> lookups -> store), vector-ALU-bound beyond.  What the split of the work does about it:
//   * prepare_ln_kernel: a wave owns whole rows, so no row sum needs a workgroup barrier and the number of workgroups is
//     rows / 8 (G = 16) instead of rows / 32.  (A workgroup that owns 32 rows and meets at five barriers: 18 us at
//     591 x 1024.)
//   * prepare_kernel: no LayerNorm, tiles of 32 rows x one group.
//   * x_hat goes to the block layout through LDS in runs of at least 8 rows x 16 bytes, i.e. whole 128-byte lines
//     wherever the tensor's rows allow it.
//   * Weights: arcq_prepare_core.h.
// FP8 operands (F8): the same work with pieces of 16 values and rows padded with zeros to 128 values.
// Arithmetic: arcq_act_quant_core.h and the stage-2 expression, unchanged -- bit-identical to the stand-alone kernels.
#include "arcq_prepare_core.h"
#include "arcq_gemm.h"

#include <algorithm>

namespace arcq {
namespace {

template <typename TIN> struct PrepTile;           // a 32-row x 64-value tile in LDS: odd dword pitch, values per 16 bytes
template <> struct PrepTile<float> { static constexpr int pitch = 65, vec = 4; };
template <> struct PrepTile<__half> { static constexpr int pitch = 33, vec = 8; };

// Stage 1 without a LayerNorm.  From a few thousand rows on fp16 input is bound by the vector ALUs (12 608 x 1 536: 17.0 us, they
// issue during 95 % of it, 78 MB = 4.6 TB/s; 12 608 x 768: 10.8 us, 8 at the rate of a copy), fp32 input by memory (12 608 x
// 1 536: 22.7 us, 116 MB = 5.1 TB/s).  A wave tile is 32 rows x ONE group; lane l owns row l / 2 and the half l % 2 of the group
// (arcq_act_quant_core.h).  Data moves through a wave-private LDS tile (rows of the tile = rows of the tensor): coalesced 16-byte
// loads in, every piece column out as one 512-byte run of the block layout.  (Lanes that load their 64 contiguous bytes
// themselves, four partial lines per instruction: 16.0 us.)
// BUILDER: a fifth wave that owns no tile builds the lookup tables while the four tile waves load their first tile and take
// its statistics.  Without it the four build the tables together before their first tile.
template <typename TIN, int BITS, bool F8, bool BUILDER>
__global__ void __launch_bounds__(64 * (kPrepWaves + (BUILDER ? 1 : 0)))
prepare_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb, char *__restrict__ x_hat, float eps,
               int rows, int G, PrepWeights w0, PrepWeights w1)
{
    constexpr int kInPitch = PrepTile<TIN>::pitch;
    constexpr int kLoads = 64 / PrepTile<TIN>::vec;        // 16-byte loads per row of the tile (8 fp16 / 16 fp32)
    constexpr int kRowsPerInstr = 64 / kLoads;             // 8 / 4
    constexpr int kIters = 32 / kRowsPerInstr;             // 4 / 8
    constexpr int kPieces = F8 ? 4 : 8;                    // 16-byte pieces of a group of x_hat
    constexpr int kOutDwords = kPieces * 4, kOutPitch = kOutDwords + 1;
    __shared__ uint32_t tiles[kPrepWaves][32 * kInPitch];
    __shared__ QuantTables tables;
    if (prep_weight_workgroup<BITS, F8>(w0, w1, tables.cb)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (BUILDER && wave == kPrepWaves) {
        build_quant_tables<BITS>(load_quant_params<BITS>(thr, cb, lane), tables, lane);
        __syncthreads();
        return;
    }
    QuantParams params{};
    if (!BUILDER && wave == 0) params = load_quant_params<BITS>(thr, cb, lane);
    const int wg = blockIdx.x - (w0.blocks + w1.blocks), wgs = gridDim.x - (w0.blocks + w1.blocks);
    const int tiles_total = ((rows + 31) / 32) * G;
    const int64_t K = static_cast<int64_t>(G) * 64;
    const int row_groups = F8 ? (G + 1) / 2 * 2 : G;       // with the padding
    const int64_t block_bytes = static_cast<int64_t>(row_groups) * kPieces * 16 * 32;
    uint32_t *tile = tiles[wave];

    uint4 raw[kIters];
    auto fetch = [&](int t) {                              // tile t = (row block t / G, group t % G); zeros past the end
        const int rb = t / G, g = t - rb * G;
        const int r0 = rb * 32 + lane / kLoads;
        const TIN *p = x + r0 * K + g * 64 + (lane % kLoads) * PrepTile<TIN>::vec;
#pragma unroll
        for (int i = 0; i < kIters; ++i)
            raw[i] = t < tiles_total && r0 + i * kRowsPerInstr < rows ? *reinterpret_cast<const uint4 *>(p + i * kRowsPerInstr * K)
                                                                      : make_uint4(0, 0, 0, 0);
    };
    fetch(wg * kPrepWaves + wave);
    BucketScale bq{};
    bool table_ok = false, tables_built = false;
    const int row = lane >> 1, half = lane & 1;
    if constexpr (!BUILDER) {
        if (wave == 0) build_quant_tables<BITS>(params, tables, lane);
        __syncthreads();
        bq = tables.geometry;
        table_ok = tables.usable != 0;
        tables_built = true;
    }
    for (int tile0 = wg * kPrepWaves; tile0 < tiles_total; tile0 += wgs * kPrepWaves) {
        const int t = tile0 + wave;
        {
            uint32_t *dst = tile + (lane / kLoads) * kInPitch + (lane % kLoads) * 4;
#pragma unroll
            for (int i = 0; i < kIters; ++i) {
                uint32_t *d = dst + i * kRowsPerInstr * kInPitch;
                d[0] = raw[i].x; d[1] = raw[i].y; d[2] = raw[i].z; d[3] = raw[i].w;
            }
        }
        __builtin_amdgcn_wave_barrier();                   // the tile is private to the wave and LDS operations execute in order
        float xv[32];
        {
            const uint32_t *src = tile + row * kInPitch + half * (32 * static_cast<int>(sizeof(TIN)) / 4);
            if constexpr (sizeof(TIN) == 4) {
#pragma unroll
                for (int j = 0; j < 32; ++j) xv[j] = __uint_as_float(src[j]);
            } else {
#pragma unroll
                for (int p = 0; p < 16; ++p) {
                    const uint32_t w = src[p];
                    xv[2 * p] = __half2float(__ushort_as_half(static_cast<unsigned short>(w & 0xffffu)));
                    xv[2 * p + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w >> 16)));
                }
            }
        }
        fetch(t + wgs * kPrepWaves);                       // the wave's next tile loads under this one's arithmetic
        float mu, var, s, sum_codes;
        group_stats32x2(xv, eps, mu, var, s);
        if (BUILDER && !tables_built) {                    // once per workgroup: the builder wave's tables are ready
            __syncthreads();
            bq = tables.geometry;
            table_ok = tables.usable != 0;
            tables_built = true;
        }
        group_codes32x2<BITS>(xv, mu, var, s, tables, bq, table_ok, sum_codes);
        const float code_mean = sum_codes * 0.015625f;
        {
            uint32_t *dst = tile + row * kOutPitch + half * (kOutDwords / 2);
            if constexpr (F8) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    uint32_t o[4];
                    xhat_fp8x16(xv, 16 * i, s, code_mean, mu, o);
#pragma unroll
                    for (int d = 0; d < 4; ++d) dst[4 * i + d] = o[d];
                }
            } else {
#pragma unroll
                for (int p = 0; p < 16; ++p) {
                    const __half2 h = __floats2half2_rn(fma_f32(s, xv[2 * p] - code_mean, mu), fma_f32(s, xv[2 * p + 1] - code_mean, mu));
                    dst[p] = *reinterpret_cast<const uint32_t *>(&h);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
        if (t < tiles_total) {
            const int rb = t / G, g = t - rb * G;
            const int r = lane & 31;
            const int nrows = min(32, rows - rb * 32);     // < 32 in a ragged last block, which is stored compactly
            char *base = x_hat + rb * block_bytes + (g * kPieces * nrows + r) * 16;
            if (r < nrows) {
#pragma unroll
                for (int j = 0; j < kPieces / 2; ++j) {    // instruction j: piece columns 2j and 2j + 1, nrows x 16 bytes each
                    const int kp = j * 2 + (lane >> 5);
                    const uint32_t *src = tile + r * kOutPitch + kp * 4;
                    store_writethrough16(base + kp * (nrows * 16), src[0], src[1], src[2], src[3]);
                    if (F8 && row_groups > G && g == G - 1) store_writethrough16(base + (kPieces + kp) * (nrows * 16), 0, 0, 0, 0);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();                   // the tile is refilled in the next iteration
    }
}

// The same for launches of a few rows, which are one chain of instructions long: eight lanes a group (FP8: four), each with the
// values of one 16-byte piece of x_hat, eight (sixteen) rows a wave, no LDS but the tables.
template <typename TIN, int BITS, bool F8>
__global__ void __launch_bounds__(64 * (kPrepWaves + 1))
prepare_few_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb, char *__restrict__ x_hat, float eps,
                   int rows, int G, PrepWeights w0, PrepWeights w1)
{
    constexpr int LANES = F8 ? 4 : 8, V = 64 / LANES, ROWS = 64 / LANES;
    constexpr int kIn = V * static_cast<int>(sizeof(TIN)) / 16;
    __shared__ QuantTables tables;
    if (prep_weight_workgroup<BITS, F8>(w0, w1, tables.cb)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (wave == kPrepWaves) {
        build_quant_tables<BITS>(load_quant_params<BITS>(thr, cb, lane), tables, lane);
        __syncthreads();
        return;
    }
    const int t = static_cast<int>(blockIdx.x - (w0.blocks + w1.blocks)) * kPrepWaves + wave;
    const int rb = t / G, g = t - rb * G;
    const int r = rb * ROWS + lane / LANES, piece = lane % LANES;
    const bool live = r < rows;
    const int64_t K = static_cast<int64_t>(G) * 64;
    const uint4 *src = reinterpret_cast<const uint4 *>(x + min(r, rows - 1) * K + g * 64 + piece * V);
    uint4 raw[kIn];
#pragma unroll
    for (int i = 0; i < kIn; ++i) raw[i] = src[i];
    float v[V];
#pragma unroll
    for (int i = 0; i < kIn; ++i) {
        const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            if constexpr (sizeof(TIN) == 2) {
                v[8 * i + 2 * d] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] & 0xffffu)));
                v[8 * i + 2 * d + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] >> 16)));
            } else {
                v[4 * i + d] = __uint_as_float(w[d]);
            }
        }
    }
    float mu, var, s, sum_codes;
    group_stats_lanes<LANES>(v, eps, lane, mu, var, s);
    __syncthreads();
    group_codes_lanes<BITS, LANES>(v, mu, var, s, tables, tables.geometry, tables.usable != 0, lane, sum_codes);
    if (!live) return;
    const float code_mean = sum_codes * 0.015625f;
    uint32_t o[4];
    if constexpr (F8) {
        xhat_fp8x16(v, 0, s, code_mean, mu, o);
    } else {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const __half2 h = __floats2half2_rn(fma_f32(s, v[2 * d] - code_mean, mu), fma_f32(s, v[2 * d + 1] - code_mean, mu));
            o[d] = *reinterpret_cast<const uint32_t *>(&h);
        }
    }
    const int blk = r >> 5, nrows = min(32, rows - blk * 32), row_groups = F8 ? (G + 1) / 2 * 2 : G;
    char *dst = x_hat + (static_cast<int64_t>(blk) * 32 * row_groups * LANES + (g * LANES + piece) * nrows + (r & 31)) * 16;
    store_writethrough16(dst, o[0], o[1], o[2], o[3]);
    if (F8 && row_groups > G && g == G - 1) store_writethrough16(dst + LANES * nrows * 16, 0, 0, 0, 0);
}

// LayerNorm over the rows first.  Wave w of a workgroup's tile takes rows R w ... R w + R - 1, 2 G lanes per row, so that the
// row sums stay inside the wave.  Vector-ALU-bound from a few thousand rows on, one dependent chain below.  The partial sums of
// a row go through wave-private LDS padded with zeros to a multiple of eight (x + 0 leaves the sum as it is), so that all reads
// of a sum are in flight together, and gamma and beta lie in LDS (pitch 36 per 32 values: conflict-free 16-byte reads).  With
// one read per loop trip and gamma / beta from L2: see the figures at the launch.
// LANES lanes a group: two, or four or eight in launches of a few rows, which are one chain of instructions long.
constexpr int gamma_pitch(int lanes) { return 64 / lanes + 4; }
// BUILDER: as above; the tables and gamma / beta are first needed behind the first tile's row sums.
template <typename TIN, int BITS, int LANES, bool BUILDER>
__global__ void __launch_bounds__(64 * (kPrepWaves + (BUILDER ? 1 : 0))) __attribute__((amdgpu_waves_per_eu(4)))
prepare_ln_kernel(const TIN *__restrict__ x, const float *__restrict__ gamma, const float *__restrict__ beta, float ln_eps,
                  const float *__restrict__ thr, const float *__restrict__ cb, char *__restrict__ x_hat, float eps, int rows,
                  int G, int R, uint32_t rw_inverse, int tiles, PrepWeights w0, PrepWeights w1)
{
    constexpr int V = 64 / LANES, kGammaPitch = gamma_pitch(LANES);    // values per lane
    constexpr int kIn = V * static_cast<int>(sizeof(TIN)) / 16;        // 16-byte loads per lane
    extern __shared__ __attribute__((aligned(16))) unsigned char prep_smem[];
    __shared__ QuantTables tables;
    if (prep_weight_workgroup<BITS, false>(w0, w1, tables.cb)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (BUILDER && wave == kPrepWaves) {
        build_quant_tables<BITS>(load_quant_params<BITS>(thr, cb, lane), tables, lane);
        __syncthreads();
        return;
    }
    QuantParams params{};
    if (!BUILDER && wave == 0) params = load_quant_params<BITS>(thr, cb, lane);
    const int wg = blockIdx.x - (w0.blocks + w1.blocks), wgs = gridDim.x - (w0.blocks + w1.blocks);
    const int P = LANES * G;                                // lanes per row
    const int rl = lane / P, pl = lane - rl * P;            // row of the wave, lane of the row
    const int K = G * 64;
    const bool lane_used = rl < R;
    const int RW = kPrepWaves * R;                          // rows of a tile
    const int chunks = (2 * G + 7) / 8;                     // of eight partial sums (32 values each)
    unsigned char *tile = prep_smem;                        // RW * G * 128 bytes
    float *part = reinterpret_cast<float *>(prep_smem + RW * G * 128) + wave * (R * chunks * 8);
    float *s_gamma = reinterpret_cast<float *>(prep_smem + RW * G * 128) + kPrepWaves * (R * chunks * 8);
    float *s_beta = s_gamma + P * kGammaPitch;

    uint4 raw[kIn];
    auto fetch = [&](int t) {
        const int row = t * RW + wave * R + rl;
        const bool valid = lane_used && t < tiles && row < rows;
        const uint4 *p = reinterpret_cast<const uint4 *>(x + static_cast<int64_t>(valid ? row : 0) * K + (valid ? pl * V : 0));
#pragma unroll
        for (int i = 0; i < kIn; ++i) raw[i] = valid ? p[i] : make_uint4(0, 0, 0, 0);
    };
    fetch(wg);
    for (int i = tid; i < K / 4; i += kPrepThreads) {
        const float4 gv = reinterpret_cast<const float4 *>(gamma)[i], bv = reinterpret_cast<const float4 *>(beta)[i];
        const int at = i / (V / 4) * kGammaPitch + i % (V / 4) * 4;
        *reinterpret_cast<float4 *>(s_gamma + at) = gv;
        *reinterpret_cast<float4 *>(s_beta + at) = bv;
    }
    for (int i = lane; i < R * chunks * 8; i += 64) part[i] = 0.0f;
    if (!BUILDER && wave == 0) build_quant_tables<BITS>(params, tables, lane);      // while the first tile is on its way
    BucketScale bq{};
    bool table_ok = false, ready = false;
    const float fk = static_cast<float>(K);
    float *my_part = part + (lane_used ? rl : 0) * (chunks * 8);
    const float *my_gamma = s_gamma + (lane_used ? pl : 0) * kGammaPitch, *my_beta = s_beta + (lane_used ? pl : 0) * kGammaPitch;

    for (int t = wg; t < tiles; t += wgs) {
        float xv[V];
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
        if (t + wgs < tiles) fetch(t + wgs);                // the next tile loads under this one's arithmetic
        // Row sums: every 32 values are folded serially, the row's 2 G partial sums are added in order (group by group, lower half
        // first) by every lane of the row.
        constexpr int kPer = LANES / 2;                     // lanes per partial sum (the last one has it)
        auto row_total = [&](float mine) {
            if (lane_used && pl % kPer == kPer - 1) my_part[pl / kPer] = mine;
            __builtin_amdgcn_wave_barrier();
            float acc = 0.0f;
            for (int c0 = 0; c0 < chunks; c0 += 4) {        // (one trip up to K = 1 024)
                float4 v[4][2];
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c0 + c < chunks) {
                        v[c][0] = *reinterpret_cast<const float4 *>(my_part + (c0 + c) * 8);
                        v[c][1] = *reinterpret_cast<const float4 *>(my_part + (c0 + c) * 8 + 4);
                    }
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c0 + c < chunks) {
#pragma unroll
                        for (int h = 0; h < 2; ++h) {
                            acc += v[c][h].x;
                            acc += v[c][h].y;
                            acc += v[c][h].z;
                            acc += v[c][h].w;
                        }
                    }
            }
            __builtin_amdgcn_wave_barrier();
            return acc;
        };
        const float mean = row_total(lanes_serial_sum<kPer>(xv)) / fk;
        float sq[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
            xv[j] -= mean;
            sq[j] = xv[j] * xv[j];
        }
        const float rstd = 1.0f / sqrtf(row_total(lanes_serial_sum<kPer>(sq)) / fk + ln_eps);
        if (!ready) {                                       // once per workgroup: the tables, gamma and beta are in LDS
            __syncthreads();
            bq = tables.geometry;
            table_ok = tables.usable != 0;
            ready = true;
        }
#pragma unroll
        for (int j4 = 0; j4 < V / 4; ++j4) {
            const float4 gv = *reinterpret_cast<const float4 *>(my_gamma + 4 * j4), bv = *reinterpret_cast<const float4 *>(my_beta + 4 * j4);
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
        float mu, var, s, sum_codes;
        if constexpr (LANES == 2) {
            group_stats32x2(xv, eps, mu, var, s);
            group_codes32x2<BITS, 0, sizeof(TIN) == 4 ? 4 : 8>(xv, mu, var, s, tables, bq, table_ok, sum_codes);      // (fp32: eight at a time spill)
        } else {
            group_stats_lanes<LANES>(xv, eps, lane, mu, var, s);
            group_codes_lanes<BITS, LANES>(xv, mu, var, s, tables, bq, table_ok, lane, sum_codes);
        }
        const float code_mean = sum_codes * 0.015625f;
        // ---- out: piece (k8, row) at LDS slot k8 * RW + row, then 16 bytes per lane, rows fastest ----
        if (lane_used) {
#pragma unroll
            for (int i = 0; i < V / 8; ++i) {
                uint32_t w[4];
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    const int j = 8 * i + 2 * d;
                    const __half2 h = __floats2half2_rn(fma_f32(s, xv[j] - code_mean, mu), fma_f32(s, xv[j + 1] - code_mean, mu));
                    w[d] = *reinterpret_cast<const uint32_t *>(&h);
                }
                *reinterpret_cast<uint4 *>(tile + ((pl * (V / 8) + i) * RW + wave * R + rl) * 16) = make_uint4(w[0], w[1], w[2], w[3]);
            }
        }
        __syncthreads();
        const int r0 = t * RW;
        const int pieces = G * 8 * RW;
        for (int p = tid; p < pieces; p += kPrepThreads) {
            const int k8 = static_cast<int>(static_cast<uint32_t>(p) * rw_inverse >> 20), r = p - k8 * RW;      // p / RW
            const int rr = r0 + r, blk = rr >> 5;
            if (rr < rows) {
                const uint4 v = *reinterpret_cast<const uint4 *>(tile + p * 16);
                const int nrows = min(32, rows - blk * 32);
                store_writethrough16(x_hat + static_cast<int64_t>(blk) * (64 * K) + (k8 * nrows + (rr & 31)) * 16, v.x, v.y, v.z, v.w);
            }
        }
        __syncthreads();
    }
}

template <typename TIN, int BITS, bool F8>
void launch_prepare_t(const arcq_prepare_args &a, float eps, const PrepWeights &w0, const PrepWeights &w1, hipStream_t stream)
{
    const int G = static_cast<int>(a.K / 64), rows = static_cast<int>(a.rows);
    const unsigned weights = w0.blocks + w1.blocks;
    const TIN *x = static_cast<const TIN *>(a.x);
    char *x_hat = static_cast<char *>(a.x_hat);
    if constexpr (!F8) {
        if (a.ln_weight && rows > 0) {
            auto run = [&](auto lanes, auto builder) {
                constexpr int LANES = decltype(lanes)::value;
                constexpr bool BUILDER = decltype(builder)::value;
                const int R = 64 / (LANES * G), RW = kPrepWaves * R, tiles = (rows + RW - 1) / RW;      // rows per wave and tile
                const size_t smem = static_cast<size_t>(RW) * G * 128 + kPrepWaves * (R * ((2 * G + 7) / 8) * 8) * 4 +
                                    static_cast<size_t>(LANES * G) * gamma_pitch(LANES) * 8;
                // Beyond four workgroups per CU the waves walk their tiles: the lookup tables are built once per workgroup.
                // (2^20 / RW rounded up: exact for all 1 024 pieces or fewer of a tile, whatever the number of groups.  The division
                // cost 20 instructions a piece: 12 608 x 1 024 16.9 -> 16.1 us)
                hipLaunchKernelGGL((prepare_ln_kernel<TIN, BITS, LANES, BUILDER>), dim3(weights + std::min(tiles, 4 * device_cus())),
                                   dim3(kPrepThreads + (BUILDER ? 64 : 0)), smem, stream, x, a.ln_weight, a.ln_bias, a.ln_eps, a.thresholds,
                                   a.codebook, x_hat, eps, rows, G, R, static_cast<uint32_t>(((1 << 20) + RW - 1) / RW), tiles, w0, w1);
            };
            using I2 = std::integral_constant<int, 2>;
            using I4 = std::integral_constant<int, 4>;
            using I8 = std::integral_constant<int, 8>;
            auto tiles_of = [&](int lanes) {
                const int RW = kPrepWaves * (64 / (lanes * G));
                return (rows + RW - 1) / RW;
            };
            // With more lanes a group while that is at most two tiles per CU: 197 x 384 6.3 -> 4.3 us with eight lanes, 2 048 x 384
            // 6.6 -> 4.7, 1 576 x 768 6.6 -> 5.4 with four; beyond, 6 304 x 384 (1 576 tiles of eight lanes) 7.4 -> 8.4.
            if (G <= 8 && tiles_of(8) <= 2 * device_cus()) run(I8{}, std::true_type{});
            else if (G <= 16 && tiles_of(4) <= 2 * device_cus()) run(I4{}, std::true_type{});
            else if (tiles_of(2) <= 2 * device_cus()) run(I2{}, std::true_type{});
            else run(I2{}, std::false_type{});
            return;
        }
    }
    // Few rows: 197 x 384 4.7 -> 3.8 us, 3 349 x 384 5.0 -> 4.6; fp32 and FP8 move other amounts and win longer (6 304 x 384 fp32
    // 7.1 -> 5.3, 6 304 x 768 FP8 8.0 -> 6.9, both 1 182 workgroups, where fp16 takes 5.5 against 5.1).
    const int few = ((rows + (F8 ? 15 : 7)) / (F8 ? 16 : 8) * G + kPrepWaves - 1) / kPrepWaves;
    if (weights + few == 0) return;
    if (few <= (F8 || sizeof(TIN) == 4 ? 6 : 4) * device_cus()) {
        hipLaunchKernelGGL((prepare_few_kernel<TIN, BITS, F8>), dim3(weights + few), dim3(kPrepThreads + 64), 0, stream, x, a.thresholds,
                           a.codebook, x_hat, eps, rows, G, w0, w1);
        return;
    }
    // Up to 2 048 tiles (two workgroups per CU) every wave takes one tile and a fifth wave builds the tables meanwhile (6 304 x 384:
    // 5.1 us).  Beyond that the grid is what the chip holds at once (fp32: three workgroups per CU; 12 608 x 1 536 25.4 -> 21.7 us
    // against four), the tables are built once per workgroup and the waves walk their tiles with the next one's loads in flight
    // (12 608 x 1 536: 18-19 us; a workgroup per four tiles 27-30).
    const int tiles = ((rows + 31) / 32) * G, wgs = std::min((tiles + kPrepWaves - 1) / kPrepWaves, (sizeof(TIN) == 4 ? 3 : 4) * device_cus());
    if constexpr (!F8) {
        if (tiles <= 2048) {
            hipLaunchKernelGGL((prepare_kernel<TIN, BITS, F8, true>), dim3(weights + wgs), dim3(kPrepThreads + 64), 0, stream, x, a.thresholds,
                               a.codebook, x_hat, eps, rows, G, w0, w1);
            return;
        }
    }
    hipLaunchKernelGGL((prepare_kernel<TIN, BITS, F8, false>), dim3(weights + wgs), dim3(kPrepThreads), 0, stream, x, a.thresholds,
                       a.codebook, x_hat, eps, rows, G, w0, w1);
}

template <typename TIN, bool F8>
void launch_prepare_bits(const arcq_prepare_args &a, float eps, const PrepWeights &w0, const PrepWeights &w1, hipStream_t stream)
{
    if (a.bits == 4) launch_prepare_t<TIN, 4, F8>(a, eps, w0, w1, stream);
    else if (a.bits == 3) launch_prepare_t<TIN, 3, F8>(a, eps, w0, w1, stream);
    else launch_prepare_t<TIN, 2, F8>(a, eps, w0, w1, stream);
}

}  // namespace
}  // namespace arcq

using namespace arcq;

static void launch_prepare(const arcq_prepare_args &a, float eps, const PrepWeights &w0, const PrepWeights &w1, hipStream_t stream)
{
    if (a.fp8) {
        if (a.x_dtype == ARCQ_F32) launch_prepare_bits<float, true>(a, eps, w0, w1, stream);
        else launch_prepare_bits<__half, true>(a, eps, w0, w1, stream);
    } else if (a.x_dtype == ARCQ_F32) {
        launch_prepare_bits<float, false>(a, eps, w0, w1, stream);
    } else {
        launch_prepare_bits<__half, false>(a, eps, w0, w1, stream);
    }
}

ARCQ_API int arcq_prepare(const arcq_prepare_args *a, void *stream)
{
    if (!a) return fail(ARCQ_ERR_NULL, "arcq_prepare: args must not be NULL");
    if (!bits_ok(a->bits)) return fail(ARCQ_ERR_BITS, "arcq_prepare: bits must be 2, 3, or 4");
    if (a->rows < 0 || a->K < 0) return fail(ARCQ_ERR_SHAPE, "arcq_prepare: bad sizes");
    PrepWeights pw[2];
    for (int i = 0; i < 2; ++i) {
        const int rc = weight_job_checked("arcq_prepare", &a->weights[i], a->fp8 != 0, pw[i]);
        if (rc != ARCQ_OK) return rc;
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
    launch_prepare(*a, 1.0e-6f, pw[0], pw[1], static_cast<hipStream_t>(stream));
    return launch_status("arcq_prepare");
}

static int act_quant_blocked(const void *x, int x_dtype, const float *thresholds, const float *codebook, void *x_hat_blocked,
                             int64_t rows, int64_t cols, int bits, float eps, const PrepWeights &w, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_act_quant_blocked: bits must be 2, 3, or 4");
    if (rows < 0 || cols < 0) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked: bad sizes");
    if (cols % 64 != 0) return fail(ARCQ_ERR_GROUP, "arcq_act_quant_blocked: in_features must be divisible by 64");
    if (x_dtype != ARCQ_F32 && x_dtype != ARCQ_F16)
        return fail(ARCQ_ERR_DTYPE, "arcq_act_quant_blocked: x must be float32 or float16");
    if (rows * cols == 0 && w.blocks == 0) return ARCQ_OK;
    if (!x || !thresholds || !codebook || !x_hat_blocked)
        return fail(ARCQ_ERR_NULL, "arcq_act_quant_blocked: x, thresholds, codebook and x_hat_blocked must not be NULL");
    if (x_hat_blocked == x) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_act_quant_blocked: x_hat_blocked must not alias x");
    if (rows * cols * 2 >= (int64_t(1) << 32)) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked: tensor too large");
    if (!aligned(x, 16) || !aligned(x_hat_blocked, 16))
        return fail(ARCQ_ERR_ALIGN, "arcq_act_quant_blocked: x and x_hat_blocked must be 16-byte aligned");
    arcq_prepare_args a = {};
    a.x_dtype = x_dtype, a.bits = bits, a.rows = rows, a.K = cols;
    a.x = x, a.thresholds = thresholds, a.codebook = codebook, a.x_hat = x_hat_blocked;
    launch_prepare(a, eps, w, PrepWeights{}, static_cast<hipStream_t>(stream));
    return launch_status("arcq_act_quant_blocked");
}

ARCQ_API int arcq_act_quant_blocked(const void *x, int x_dtype, const float *thresholds, const float *codebook,
                                    void *x_hat_blocked, int64_t rows, int64_t cols, int bits, float eps, void *stream)
{
    return act_quant_blocked(x, x_dtype, thresholds, codebook, x_hat_blocked, rows, cols, bits, eps, PrepWeights{}, stream);
}

// Stage 1 into the block layout and, in the same launch, w_hat[N, cols] (fp16, group size 64) from the layer's packed
// weights: the two inputs of the copying GEMM variant.
ARCQ_API int arcq_act_quant_blocked_with_weights(const void *x, int x_dtype, const float *thresholds,
                                                 const float *codebook, void *x_hat_blocked, int64_t rows, int64_t cols,
                                                 int bits, float eps, const uint8_t *packed_w, const float *w_codebook,
                                                 const float *w_center, const float *w_scale, const float *w_code_sum,
                                                 void *w_hat, int64_t N, void *stream)
{
    if (N < 0) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked_with_weights: bad sizes");
    if (N == 0 || cols <= 0 || cols % 64 != 0)      // no weights to rebuild (or sizes the plain entry point reports)
        return arcq_act_quant_blocked(x, x_dtype, thresholds, codebook, x_hat_blocked, rows, cols, bits, eps, stream);
    if (!packed_w || !w_codebook || !w_center || !w_scale || !w_code_sum || !w_hat)
        return fail(ARCQ_ERR_NULL, "arcq_act_quant_blocked_with_weights: NULL weight tensor pointer");
    if (!aligned(w_hat, 16) || !aligned(packed_w, 4))
        return fail(ARCQ_ERR_ALIGN, "arcq_act_quant_blocked_with_weights: w_hat must be 16-byte, packed_w 4-byte aligned");
    if (N * cols >= (int64_t(1) << 31))
        return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked_with_weights: weight tensor too large");
    const arcq_prepare_weights w = {packed_w, w_codebook, w_center, w_scale, w_code_sum, w_hat, N, cols, 1, 1.0f};
    return act_quant_blocked(x, x_dtype, thresholds, codebook, x_hat_blocked, rows, cols, bits, eps, weight_job(w, false), stream);
}

// LayerNorm (weight ln_weight[cols], bias ln_bias[cols], fp32) followed by stage 1 into the block layout, in one
// launch; optionally (packed_w != NULL) the same launch reconstructs w_hat[N, cols] as
// arcq_act_quant_blocked_with_weights does.  cols / 64 must be between 1 and 16.
ARCQ_API int arcq_act_quant_blocked_ln(const void *x, int x_dtype, const float *ln_weight, const float *ln_bias, float ln_eps,
                                       const float *thresholds, const float *codebook, void *x_hat_blocked,
                                       int64_t rows, int64_t cols, int bits, float eps,
                                       const uint8_t *packed_w, const float *w_codebook, const float *w_center,
                                       const float *w_scale, const float *w_code_sum, void *w_hat, int64_t N, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_act_quant_blocked_ln: bits must be 2, 3, or 4");
    if (rows < 0 || cols < 0 || N < 0) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked_ln: bad sizes");
    if (cols % 64 != 0) return fail(ARCQ_ERR_GROUP, "arcq_act_quant_blocked_ln: in_features must be divisible by 64");
    if (cols < 64 || cols > 1024)
        return fail(ARCQ_ERR_UNSUPPORTED, "arcq_act_quant_blocked_ln: in_features must be between 64 and 1024 (got %lld)",
                    static_cast<long long>(cols));
    if (x_dtype != ARCQ_F32 && x_dtype != ARCQ_F16)
        return fail(ARCQ_ERR_DTYPE, "arcq_act_quant_blocked_ln: x must be float32 or float16");
    PrepWeights w{};
    if (packed_w && N > 0) {
        if (!w_codebook || !w_center || !w_scale || !w_code_sum || !w_hat)
            return fail(ARCQ_ERR_NULL, "arcq_act_quant_blocked_ln: NULL weight tensor pointer");
        if (!aligned(w_hat, 16) || !aligned(packed_w, 4))
            return fail(ARCQ_ERR_ALIGN, "arcq_act_quant_blocked_ln: w_hat must be 16-byte, packed_w 4-byte aligned");
        if (N * cols >= (int64_t(1) << 31)) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked_ln: weight tensor too large");
        w = weight_job({packed_w, w_codebook, w_center, w_scale, w_code_sum, w_hat, N, cols, 1, 1.0f}, false);
    }
    if (rows == 0 && w.blocks == 0) return ARCQ_OK;
    if (!x || !ln_weight || !ln_bias || !thresholds || !codebook || !x_hat_blocked)
        return fail(ARCQ_ERR_NULL, "arcq_act_quant_blocked_ln: x, ln_weight, ln_bias, thresholds, codebook and x_hat_blocked must not be NULL");
    if (x_hat_blocked == x) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_act_quant_blocked_ln: x_hat_blocked must not alias x");
    if (rows * cols * 2 >= (int64_t(1) << 32)) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant_blocked_ln: tensor too large");
    if (!aligned(x, 16) || !aligned(x_hat_blocked, 16) || !aligned(ln_weight, 16) || !aligned(ln_bias, 16))
        return fail(ARCQ_ERR_ALIGN, "arcq_act_quant_blocked_ln: x, x_hat_blocked, ln_weight and ln_bias must be 16-byte aligned");
    arcq_prepare_args a = {};
    a.x_dtype = x_dtype, a.bits = bits, a.rows = rows, a.K = cols;
    a.ln_weight = ln_weight, a.ln_bias = ln_bias, a.ln_eps = ln_eps;
    a.x = x, a.thresholds = thresholds, a.codebook = codebook, a.x_hat = x_hat_blocked;
    launch_prepare(a, eps, w, PrepWeights{}, static_cast<hipStream_t>(stream));
    return launch_status("arcq_act_quant_blocked_ln");
}
