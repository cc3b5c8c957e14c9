// Stage 1: activation group-residual quantizer (semantics:
// EXT/arcq_activation_kernel.cu:24-184; fused quantize+reconstruct as in
// FQ/arcq_packed_triton.py:123-178).
//
// Per group of gs input channels of one token:
//   mu = (x0 + x1 + ... ) / gs           serial, left to right
//   s  = sqrt((sum_j (x_j - mu)^2) / gs + eps)
//   t_j = (x_j - mu) / s                 correctly rounded
//   code_j = number of leading thresholds with t_j > thr[i]
//   S = sum_j cb[code_j]                 serial
//   x_hat_j = fma(s, cb[code_j] - S/gs, mu)
//
// gs == 64 kernel.  x is [rows, G*64], so the groups of the whole tensor are consecutive 64-element
// runs of one flat array.  A wave owns a tile of 64 consecutive groups and gives every lane ONE group,
// so the serial sums are plain register loops (64 independent chains per wave).  Data moves between
// the coalesced global layout (16-byte accesses) and the lane-per-group layout through a per-wave LDS
// tile whose row stride is odd in dwords (33 for fp16, 65 for fp32), which makes both the row-wise
// 16-byte phase and the per-lane column phase bank-conflict free.
//
// Two things keep the per-element VALU work low without changing a single result bit:
//  * t = d/s is not formed.  Whether RN(d/s) lies above a threshold is the sign of a remainder, two fused operations; groups
//    whose s or mu fall outside the range where that is exact take the plain division and a bisection over the thresholds.
//  * the threshold search is one table lookup and one such sign: d times an approximate 1/s names one of up to 513 buckets over
//    [-8, 8] (|t| <= 8 always, since s^2 >= d_j^2/64; the bucket width adapts to the smallest gap between thresholds); a bucket
//    stores how many thresholds lie in lower buckets and the single threshold inside it.  Thresholds keep a margin from the
//    buckets' edges, so the neighbouring bucket that the approximate quotient may name gives the same code.  The codebook
//    lies in LDS once: a read of sixteen different entries meets no bank twice.  If two thresholds share a bucket, one lies
//    outside [-8, 8) or at an edge both ways, or they are not sorted, that is how all codes are found.
// The arithmetic itself lives in arcq_act_quant_core.h (shared with the fused small-M layer kernel).
#include "arcq_act_quant_core.h"
#include "arcq_gemm.h"

#include <algorithm>

namespace arcq {

constexpr int kWaves = 4;          // waves (tiles in flight) per workgroup
constexpr int kTileGroups = 64;    // groups per tile = lanes per wave
template <typename T> struct Tile;
template <> struct Tile<float> { static constexpr int stride = 65; static constexpr int vec = 4; };
template <> struct Tile<__half> { static constexpr int stride = 33; static constexpr int vec = 8; };

// Coalesced 16-byte global loads of one tile (64 groups x 64 elements) into registers, and from there
// into the wave's LDS tile.  Two steps so that the first tile's loads can be in flight during the
// per-workgroup setup.
template <typename TIN> struct TileRegs { uint4 raw[kTileGroups * 64 / (64 * Tile<TIN>::vec)]; };

template <typename TIN>
__device__ __forceinline__ void fetch_tile(const TIN *__restrict__ x, int64_t elem0, int64_t elem_end,
                                           TileRegs<TIN> &r, int lane)
{
    constexpr int n = Tile<TIN>::vec;
    constexpr int iters = kTileGroups * 64 / (64 * n);
#pragma unroll
    for (int i = 0; i < iters; ++i) {
        const int e = (i * 64 + lane) * n;
        r.raw[i] = (elem0 + e < elem_end) ? *reinterpret_cast<const uint4 *>(x + elem0 + e) : make_uint4(0, 0, 0, 0);
    }
}

template <typename TIN>
__device__ __forceinline__ void commit_tile(const TileRegs<TIN> &r, uint32_t *__restrict__ tile, int lane)
{
    constexpr int n = Tile<TIN>::vec;
    constexpr int iters = kTileGroups * 64 / (64 * n);
#pragma unroll
    for (int i = 0; i < iters; ++i) {
        const int e = (i * 64 + lane) * n;
        uint32_t *dst = tile + (e >> 6) * Tile<TIN>::stride + (e & 63) * static_cast<int>(sizeof(TIN)) / 4;
        dst[0] = r.raw[i].x; dst[1] = r.raw[i].y; dst[2] = r.raw[i].z; dst[3] = r.raw[i].w;
    }
}

template <typename TOUT>
__device__ __forceinline__ void store_tile(TOUT *__restrict__ out, int64_t elem0, int64_t elem_end,
                                           const uint32_t *__restrict__ tile, int lane)
{
    constexpr int n = Tile<TOUT>::vec;
    constexpr int iters = kTileGroups * 64 / (64 * n);
#pragma unroll
    for (int i = 0; i < iters; ++i) {
        const int e = (i * 64 + lane) * n;
        if (elem0 + e >= elem_end) continue;
        const uint32_t *src = tile + (e >> 6) * Tile<TOUT>::stride + (e & 63) * static_cast<int>(sizeof(TOUT)) / 4;
        *reinterpret_cast<uint4 *>(out + elem0 + e) = make_uint4(src[0], src[1], src[2], src[3]);
    }
}

// The lane's own group (row `lane` of the tile) as 64 floats.
template <typename TIN>
__device__ __forceinline__ void read_row(const uint32_t *__restrict__ row, float (&v)[64])
{
    if constexpr (sizeof(TIN) == 4) {
#pragma unroll
        for (int j = 0; j < 64; ++j) v[j] = __uint_as_float(row[j]);
    } else {
#pragma unroll
        for (int p = 0; p < 32; ++p) {
            const uint32_t w = row[p];
            v[2 * p] = __half2float(__ushort_as_half(static_cast<unsigned short>(w & 0xffffu)));
            v[2 * p + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w >> 16)));
        }
    }
}

template <typename TOUT>
__device__ __forceinline__ void write_row(uint32_t *__restrict__ row, const float (&v)[64])
{
    if constexpr (sizeof(TOUT) == 4) {
#pragma unroll
        for (int j = 0; j < 64; ++j) row[j] = __float_as_uint(v[j]);
    } else {
#pragma unroll
        for (int p = 0; p < 32; ++p) {
            const __half2 h = __floats2half2_rn(v[2 * p], v[2 * p + 1]);
            row[p] = *reinterpret_cast<const uint32_t *>(&h);
        }
    }
}

// The 64 codes, a byte each, as packed dwords, LSB first.
template <int BITS>
__device__ __forceinline__ void pack64(const uint32_t (&c)[16], uint32_t (&w)[2 * BITS])
{
    uint32_t four[16];      // 4 BITS bits each
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        constexpr uint32_t mask = (1u << BITS) - 1;
        four[k] = c[k] & mask;
#pragma unroll
        for (int q = 1; q < 4; ++q) four[k] |= (c[k] >> (q * (8 - BITS))) & (mask << (q * BITS));
    }
    if constexpr (BITS == 4 || BITS == 2) {
        constexpr int per = 8 / BITS;
#pragma unroll
        for (int d = 0; d < 2 * BITS; ++d) {
            uint32_t v = four[d * per];
#pragma unroll
            for (int q = 1; q < per; ++q) v |= four[d * per + q] << (4 * BITS * q);
            w[d] = v;
        }
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) {      // 8 codes -> one 24-bit chunk; 4 chunks -> 3 dwords
            uint32_t ch[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) ch[k] = four[8 * h + 2 * k] | four[8 * h + 2 * k + 1] << 12;
            w[3 * h + 0] = ch[0] | (ch[1] << 24);
            w[3 * h + 1] = (ch[1] >> 8) | (ch[2] << 16);
            w[3 * h + 2] = (ch[2] >> 16) | (ch[3] << 8);
        }
    }
}

// CODES = false drops everything only the code outputs need (the on-the-fly layer asks for x_hat alone).  The codes of a group stay a
// byte each in sixteen registers, so that two waves share a SIMD in every form (a register for each code: 300 of them and one wave;
// packed codes and x_hat of 12 608 x 1 536 fp32 42.6 us, 49.5 with all lookups in flight, 30.6 now).
template <typename TIN, typename TOUT, int BITS, bool CODES>
__global__ void __launch_bounds__(64 * kWaves, 2)
act_quant_g64_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb,
                     uint8_t *__restrict__ packed, uint8_t *__restrict__ codes_u8,
                     float *__restrict__ center, float *__restrict__ scale, float *__restrict__ code_sum,
                     TOUT *__restrict__ x_hat, int64_t total_groups, float eps)
{
    constexpr int L = 1 << BITS;
    constexpr int kStride = (Tile<TIN>::stride > Tile<TOUT>::stride) ? Tile<TIN>::stride : Tile<TOUT>::stride;
    __shared__ uint32_t tiles[kWaves][kTileGroups * kStride];
    __shared__ QuantTables tables;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;

    QuantParams params{};
    if (wave == 0) params = load_quant_params<BITS>(thr, cb, lane);
    // The first tile of this wave is requested before anything else: its latency overlaps the setup below.
    const int64_t ntiles = (total_groups + kTileGroups - 1) / kTileGroups;
    const int64_t elem_end = total_groups * 64;
    TileRegs<TIN> regs;
    {
        const int64_t first = static_cast<int64_t>(blockIdx.x) * kWaves + wave;
        fetch_tile<TIN>(x, first * kTileGroups * 64, elem_end, regs, lane);      // zero-fills past the end
    }

    // The lookup tables are built once per workgroup, before the first tile's values are unpacked into registers.
    // (Built between the two halves of the first tile, or with both orders in the kernel and a flag to choose, the
    // variants that write codes run 20-40 % slower: registers.)
    if (wave == 0) build_quant_tables<BITS>(params, tables, lane);
    __syncthreads();
    const BucketScale bq = tables.geometry;
    const bool table_ok = tables.usable != 0;

    uint32_t *tile = tiles[wave];

    // All four waves run the same number of iterations so that the barriers below are uniform.
    const int64_t tile_step = static_cast<int64_t>(gridDim.x) * kWaves;
    for (int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kWaves; tile0 < ntiles; tile0 += tile_step) {
        const int64_t group0 = (tile0 + wave) * kTileGroups;
        const int64_t elem0 = group0 * 64;
        commit_tile<TIN>(regs, tile, lane);
        __syncthreads();

        float xv[64];
        read_row<TIN>(tile + lane * Tile<TIN>::stride, xv);
        // The wave's next tile (zeros past the end) loads under this one's arithmetic.
        fetch_tile<TIN>(x, (group0 + tile_step * kTileGroups) * 64, elem_end, regs, lane);

        float mu, var, s, sum_codes;
        uint32_t code[CODES ? 16 : 1];
        group_stats64(xv, eps, mu, var, s);
        // (eight lookups in flight: with all 64 the compiler delays the sums, x_hat of 12 608 x 1 536 fp32 32.9 us against 28.3)
        group_codes64<BITS, CODES, 8>(xv, mu, var, s, tables, bq, table_ok, sum_codes, code);

        const int64_t g = group0 + lane;
        if (g < total_groups) {
            if (center) center[g] = mu;
            if (scale) scale[g] = s;
            if (code_sum) code_sum[g] = sum_codes;
            if constexpr (CODES) {
                if (packed) {
                    uint32_t w[2 * BITS];
                    pack64<BITS>(code, w);
                    uint32_t *dst = reinterpret_cast<uint32_t *>(packed + g * (8 * BITS));
                    if constexpr (BITS == 4) {
                        reinterpret_cast<uint4 *>(dst)[0] = make_uint4(w[0], w[1], w[2], w[3]);
                        reinterpret_cast<uint4 *>(dst)[1] = make_uint4(w[4], w[5], w[6], w[7]);
                    } else if constexpr (BITS == 2) {
                        reinterpret_cast<uint4 *>(dst)[0] = make_uint4(w[0], w[1], w[2], w[3]);
                    } else {
#pragma unroll
                        for (int q = 0; q < 3; ++q)
                            reinterpret_cast<uint2 *>(dst)[q] = make_uint2(w[2 * q], w[2 * q + 1]);
                    }
                }
                if (codes_u8) {
                    uint4 *dst = reinterpret_cast<uint4 *>(codes_u8 + g * 64);
#pragma unroll
                    for (int q = 0; q < 4; ++q) dst[q] = make_uint4(code[4 * q], code[4 * q + 1], code[4 * q + 2], code[4 * q + 3]);
                }
            }
        }

        if (x_hat) {
            const float code_mean = sum_codes * 0.015625f;
#pragma unroll
            for (int j = 0; j < 64; ++j) xv[j] = fma_f32(s, xv[j] - code_mean, mu);
            // Every lane has consumed its input row (program order within the wave), so rows may be
            // rewritten now, possibly with a different stride.
            write_row<TOUT>(tile + lane * Tile<TOUT>::stride, xv);
            __syncthreads();
            store_tile<TOUT>(x_hat, elem0, elem_end, tile, lane);
        }
        __syncthreads();   // the tile is reloaded in the next iteration
    }
}

// Codes and metadata, no x_hat (the encoding direction): memory-bound.  A wave tile is 32 consecutive groups, which are
// contiguous in the row-major tensor; two lanes share a group (arcq_act_quant_core.h), the inputs are loaded coalesced and
// change places in a wave-private LDS tile, and lane l's 32 codes lie at l times their size behind the tile's first: every
// store of the wave is one contiguous run.  The waves walk their tiles with the next one's loads in flight.  (A lane per group,
// act_quant_g64_kernel, when it took 297 registers: 12 608 x 1 536 fp32 at four bits 31.7 us against 19.1; 18.4 at the copy rate.)
// BUILDER as in prepare_kernel: a fifth wave builds the lookup tables of a workgroup whose waves have one tile each.
template <typename TIN, int BITS, bool BYTES, bool BUILDER>
__global__ void __launch_bounds__(64 * (kWaves + (BUILDER ? 1 : 0)))
act_quant_codes_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb,
                       uint8_t *__restrict__ codes, float *__restrict__ center, float *__restrict__ scale, float *__restrict__ code_sum,
                       int64_t total_groups, float eps)
{
    constexpr int L = 1 << BITS;
    constexpr int kPitch = Tile<TIN>::stride, kVec = Tile<TIN>::vec;
    constexpr int kLoads = 64 / kVec, kIters = 32 / kVec;              // 16-byte loads per group, per lane and tile
    constexpr int kCodeBits = BYTES ? 8 : BITS;
    __shared__ uint32_t tiles[kWaves][32 * kPitch];
    __shared__ QuantTables tables;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (BUILDER && wave == kWaves) {
        build_quant_tables<BITS>(load_quant_params<BITS>(thr, cb, lane), tables, lane);
        __syncthreads();
        return;
    }
    QuantParams params{};
    if (!BUILDER && wave == 0) params = load_quant_params<BITS>(thr, cb, lane);
    const int64_t ntiles = (total_groups + 31) / 32, step = static_cast<int64_t>(gridDim.x) * kWaves;
    uint32_t *tile = tiles[wave];
    uint4 raw[kIters];
    auto fetch = [&](int64_t t) {                                      // zeros past the end
        const int64_t g = t * 32 + lane / kLoads;
        const TIN *p = x + t * 2048 + lane * kVec;
#pragma unroll
        for (int i = 0; i < kIters; ++i)
            raw[i] = g + i * (64 / kLoads) < total_groups ? *reinterpret_cast<const uint4 *>(p + i * 64 * kVec) : make_uint4(0, 0, 0, 0);
    };
    int64_t t = static_cast<int64_t>(blockIdx.x) * kWaves + wave;
    fetch(t);
    BucketScale bq{};
    bool table_ok = false, tables_built = false;
    if constexpr (!BUILDER) {
        if (wave == 0) build_quant_tables<BITS>(params, tables, lane);
        __syncthreads();
        bq = tables.geometry;
        table_ok = tables.usable != 0;
        tables_built = true;
    }
    const int row = lane >> 1, half = lane & 1;
    for (int64_t tile0 = static_cast<int64_t>(blockIdx.x) * kWaves; tile0 < ntiles; tile0 += step, t += step) {
        {
            uint32_t *dst = tile + (lane / kLoads) * kPitch + (lane % kLoads) * 4;
#pragma unroll
            for (int i = 0; i < kIters; ++i) {
                uint32_t *d = dst + i * (64 / kLoads) * kPitch;
                d[0] = raw[i].x; d[1] = raw[i].y; d[2] = raw[i].z; d[3] = raw[i].w;
            }
        }
        __builtin_amdgcn_wave_barrier();                               // wave-private: LDS operations execute in order
        float xv[32];
        {
            const uint32_t *src = tile + row * kPitch + half * (32 * static_cast<int>(sizeof(TIN)) / 4);
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
        __builtin_amdgcn_wave_barrier();
        fetch(t + step);
        float mu, var, s, sum_codes;
        group_stats32x2(xv, eps, mu, var, s);
        if (BUILDER && !tables_built) {
            __syncthreads();
            bq = tables.geometry;
            table_ok = tables.usable != 0;
            tables_built = true;
        }
        uint32_t w[kCodeBits];
        group_codes32x2<BITS, kCodeBits>(xv, mu, var, s, tables, bq, table_ok, sum_codes, w);
        const int64_t g = t * 32 + row;
        if (t < ntiles && g < total_groups) {
            uint8_t *dst = codes + (t * 64 + lane) * (4 * kCodeBits);
#pragma unroll
            for (int d = 0; d + 4 <= kCodeBits; d += 4) *reinterpret_cast<uint4 *>(dst + 4 * d) = make_uint4(w[d], w[d + 1], w[d + 2], w[d + 3]);
            if constexpr (kCodeBits == 3) *reinterpret_cast<uint3 *>(dst) = make_uint3(w[0], w[1], w[2]);
            if constexpr (kCodeBits == 2) *reinterpret_cast<uint2 *>(dst) = make_uint2(w[0], w[1]);
            if (half == 0) {
                if (center) center[g] = mu;
                if (scale) scale[g] = s;
                if (code_sum) code_sum[g] = sum_codes;
            }
        }
    }
}

// Small launches, x_hat only: two lanes per group, no LDS tile.  When the tensor is too small to fill the chip
// (a few hundred rows) the launch lasts as long as one lane's instruction chain, so the group is shared by two lanes
// (arcq_act_quant_core.h: half the per-element work per lane, the serial sums in two linked phases, same bits).  A
// lane's 32 inputs are contiguous and consecutive lanes hold consecutive halves, so plain 16-byte loads and stores
// are already coalesced.  Every lane reads all its inputs before it writes, so x_hat may alias x.  A fifth wave builds the
// lookup tables (built by the first one under its own loads: 197 x 384 fp32 at two bits 5.6 us against 4.9).
template <typename TIN, typename TOUT, int BITS>
__global__ void __launch_bounds__(64 * (kWaves + 1))
act_quant_small_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb,
                       TOUT *__restrict__ x_hat, int64_t total_groups, float eps)
{
    constexpr int kIn = 32 * sizeof(TIN) / 16, kOut = 32 * sizeof(TOUT) / 16;
    __shared__ QuantTables tables;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    if (tid >= 64 * kWaves) {
        build_quant_tables<BITS>(load_quant_params<BITS>(thr, cb, lane), tables, lane);
        __syncthreads();
        return;
    }
    const int64_t f = (static_cast<int64_t>(blockIdx.x) * kWaves + (tid >> 6)) * 32 + (lane >> 1);   // this lane's group
    const bool valid = f < total_groups;
    const int64_t e0 = f * 64 + (lane & 1) * 32;                                                    // its first element

    uint4 raw[kIn];
#pragma unroll
    for (int i = 0; i < kIn; ++i)
        raw[i] = valid ? reinterpret_cast<const uint4 *>(x + e0)[i] : make_uint4(0, 0, 0, 0);

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
    float mu, var, s, sum_codes;
    group_stats32x2(xv, eps, mu, var, s);
    __syncthreads();
    group_codes32x2<BITS>(xv, mu, var, s, tables, tables.geometry, tables.usable != 0, sum_codes);
    const float code_mean = sum_codes * 0.015625f;
#pragma unroll
    for (int j = 0; j < 32; ++j) xv[j] = fma_f32(s, xv[j] - code_mean, mu);
    if (!valid) return;
    uint4 *dst = reinterpret_cast<uint4 *>(x_hat + e0);
    if constexpr (sizeof(TOUT) == 2) {
#pragma unroll
        for (int i = 0; i < kOut; ++i) {
            uint32_t w[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const __half2 h = __floats2half2_rn(xv[i * 8 + 2 * d], xv[i * 8 + 2 * d + 1]);
                w[d] = *reinterpret_cast<const uint32_t *>(&h);
            }
            store_writethrough16(dst + i, w[0], w[1], w[2], w[3]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < kOut; ++i)
            store_writethrough16(dst + i, __float_as_uint(xv[4 * i]), __float_as_uint(xv[4 * i + 1]),
                                 __float_as_uint(xv[4 * i + 2]), __float_as_uint(xv[4 * i + 3]));
    }
}

// Any group size: one thread per group, straight from global memory.  Slow
// (strided reads) but has no layout assumptions; used when gs != 64 or the
// pointers are not 16-byte aligned.
template <typename TIN, typename TOUT>
__global__ void __launch_bounds__(128)
act_quant_generic_kernel(const TIN *__restrict__ x, const float *__restrict__ thr, const float *__restrict__ cb,
                         uint8_t *__restrict__ packed, uint8_t *__restrict__ codes_u8,
                         float *__restrict__ center, float *__restrict__ scale, float *__restrict__ code_sum,
                         TOUT *__restrict__ x_hat, int64_t total_groups, int64_t groups_per_row,
                         int bits, int gs, float eps)
{
    const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (g >= total_groups) return;
    const int levels = 1 << bits;
    const int64_t row = g / groups_per_row;
    const int64_t gi = g - row * groups_per_row;
    const int64_t cols = groups_per_row * gs;
    const TIN *__restrict__ xg = x + g * gs;
    const float fgs = static_cast<float>(gs);

    float mu = 0.0f;
    for (int j = 0; j < gs; ++j) mu += to_float(xg[j]);
    mu /= fgs;
    float var = 0.0f;
    for (int j = 0; j < gs; ++j) {
        const float d = to_float(xg[j]) - mu;
        var += d * d;
    }
    const float s = sqrtf(var / fgs + eps);

    // Packed bytes of this group start at a byte boundary (checked on the host).
    uint8_t *pk = packed ? packed + row * packed_cols(cols, bits) + (gi * gs * bits) / 8 : nullptr;
    uint32_t acc = 0;
    int nacc = 0;
    float sum_codes = 0.0f;
    for (int j = 0; j < gs; ++j) {
        const float t = (to_float(xg[j]) - mu) / s;
        int c = 0;
        while (c < levels - 1 && t > thr[c]) ++c;
        sum_codes += cb[c];
        if (codes_u8) codes_u8[g * gs + j] = static_cast<uint8_t>(c);
        if (pk) {
            acc |= static_cast<uint32_t>(c) << nacc;
            nacc += bits;
            while (nacc >= 8) {
                *pk++ = static_cast<uint8_t>(acc & 0xffu);
                acc >>= 8;
                nacc -= 8;
            }
        }
    }
    if (center) center[g] = mu;
    if (scale) scale[g] = s;
    if (code_sum) code_sum[g] = sum_codes;
    if (x_hat) {
        // The codes are recomputed instead of stored: x_hat may alias x, so x is
        // re-read only at an index that has not been overwritten yet.
        const float code_mean = sum_codes / fgs;
        for (int j = 0; j < gs; ++j) {
            const float t = (to_float(xg[j]) - mu) / s;
            int c = 0;
            while (c < levels - 1 && t > thr[c]) ++c;
            x_hat[g * gs + j] = from_float<TOUT>(fma_f32(s, cb[c] - code_mean, mu));
        }
    }
}

template <typename TIN, typename TOUT>
static int launch(const void *x, const float *thr, const float *cb, uint8_t *packed, uint8_t *codes_u8,
                  float *center, float *scale, float *code_sum, void *x_hat,
                  int64_t rows, int64_t cols, int bits, int gs, float eps, hipStream_t stream)
{
    const int64_t groups_per_row = cols / gs;
    const int64_t total_groups = rows * groups_per_row;
    const TIN *xin = static_cast<const TIN *>(x);
    TOUT *xo = static_cast<TOUT *>(x_hat);
    const bool fast = gs == 64 && aligned(x, 16) && aligned(x_hat, 16) && aligned(packed, 16) && aligned(codes_u8, 16);
    // Fewer 64-group tiles than SIMDs and nothing but x_hat wanted: the two-lanes-per-group kernel.
    if (fast && x_hat && !packed && !codes_u8 && !center && !scale && !code_sum && total_groups <= 1024 * 64) {
        const unsigned blocks = static_cast<unsigned>((total_groups + 32 * kWaves - 1) / (32 * kWaves));
#define ARCQ_LAUNCH_SMALL(B) \
    hipLaunchKernelGGL((act_quant_small_kernel<TIN, TOUT, B>), dim3(blocks), dim3(64 * (kWaves + 1)), 0, stream, xin, thr, cb, xo, \
                       total_groups, eps)
        if (bits == 4) ARCQ_LAUNCH_SMALL(4);
        else if (bits == 3) ARCQ_LAUNCH_SMALL(3);
        else ARCQ_LAUNCH_SMALL(2);
#undef ARCQ_LAUNCH_SMALL
    } else if (fast && !x_hat && (packed != nullptr) != (codes_u8 != nullptr)) {
        // The grid is what the chip holds at once (fp32: three workgroups per CU, by their LDS and registers; a fourth that starts
        // behind them costs 15 %); one tile per wave up to 2 048 tiles (a fifth wave per workgroup builds the tables then).
        // fp32, four bits, codes and metadata: 12 608 x 1 536 31.7 -> 19.1 us, 50 432 x 1 024 71 -> 41, 394 x 768 7.5 -> 5.3.
        const int64_t ntiles = (total_groups + 31) / 32, want = (ntiles + kWaves - 1) / kWaves;
        const unsigned blocks = static_cast<unsigned>(std::min<int64_t>(want, (sizeof(TIN) == 4 ? 3 : 4) * device_cus()));
        uint8_t *codes = packed ? packed : codes_u8;
#define ARCQ_LAUNCH_CODES(B, Y)                                                                                                        \
    do {                                                                                                                               \
        if (ntiles <= 2048)                                                                                                            \
            hipLaunchKernelGGL((act_quant_codes_kernel<TIN, B, Y, true>), dim3(blocks), dim3(64 * (kWaves + 1)), 0, stream, xin, thr,   \
                               cb, codes, center, scale, code_sum, total_groups, eps);                                                  \
        else                                                                                                                           \
            hipLaunchKernelGGL((act_quant_codes_kernel<TIN, B, Y, false>), dim3(blocks), dim3(64 * kWaves), 0, stream, xin, thr, cb,    \
                               codes, center, scale, code_sum, total_groups, eps);                                                      \
    } while (0)
        if (bits == 4) { if (packed) ARCQ_LAUNCH_CODES(4, false); else ARCQ_LAUNCH_CODES(4, true); }
        else if (bits == 3) { if (packed) ARCQ_LAUNCH_CODES(3, false); else ARCQ_LAUNCH_CODES(3, true); }
        else { if (packed) ARCQ_LAUNCH_CODES(2, false); else ARCQ_LAUNCH_CODES(2, true); }
#undef ARCQ_LAUNCH_CODES
    } else if (fast) {
        const int64_t ntiles = (total_groups + kTileGroups - 1) / kTileGroups;
        // Up to 3 workgroups fit a CU (LDS); more tiles than that are walked by the grid-stride loop.
        const int64_t want = (ntiles + kWaves - 1) / kWaves;
        // The kernel holds a whole group per lane (two waves per SIMD): 512 workgroups are what the chip runs at once,
        // and a launch with more tiles than that walks them (the next tile's loads in flight) instead of starting a
        // workgroup per four tiles.  With the tables built first: packed codes + metadata from fp32 19.3 -> 16.3 us
        // at 12 608 x 384, 47 -> 32 at K = 1 536, 113 -> 71 at 50 432 x 1 024; x_hat alone 10.2 -> 10.8, 24.5 -> 22.2,
        // 53 -> 51.5.
        const int64_t cap = 512;
        const unsigned blocks = static_cast<unsigned>(want < cap ? want : cap);
        const bool codes = packed || codes_u8;
#define ARCQ_LAUNCH_G64(B, C)                                                                                     \
    hipLaunchKernelGGL((act_quant_g64_kernel<TIN, TOUT, B, C>), dim3(blocks), dim3(64 * kWaves), 0, stream, xin, \
                       thr, cb, packed, codes_u8, center, scale, code_sum, xo, total_groups, eps)
        if (bits == 4) { if (codes) ARCQ_LAUNCH_G64(4, true); else ARCQ_LAUNCH_G64(4, false); }
        else if (bits == 3) { if (codes) ARCQ_LAUNCH_G64(3, true); else ARCQ_LAUNCH_G64(3, false); }
        else { if (codes) ARCQ_LAUNCH_G64(2, true); else ARCQ_LAUNCH_G64(2, false); }
#undef ARCQ_LAUNCH_G64
    } else {
        if (packed && (static_cast<int64_t>(gs) * bits) % 8 != 0)
            return fail(ARCQ_ERR_UNSUPPORTED,
                        "arcq_act_quant: packed output needs group_size*bits divisible by 8 (got %d*%d)", gs, bits);
        const unsigned blocks = static_cast<unsigned>((total_groups + 127) / 128);
        hipLaunchKernelGGL((act_quant_generic_kernel<TIN, TOUT>), dim3(blocks), dim3(128), 0, stream, xin, thr, cb,
                           packed, codes_u8, center, scale, code_sum, xo, total_groups, groups_per_row, bits, gs, eps);
    }
    return launch_status("arcq_act_quant");
}

}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_act_quant(const void *x, int x_dtype, const float *thresholds, const float *codebook,
                            uint8_t *packed, uint8_t *codes_u8, float *center, float *scale, float *code_sum,
                            void *x_hat, int x_hat_dtype,
                            int64_t rows, int64_t cols, int bits, int group_size, float eps, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_act_quant: bits must be 2, 3, or 4");
    if (rows < 0 || cols < 0 || group_size <= 0) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant: bad sizes");
    if (cols % group_size != 0)
        return fail(ARCQ_ERR_GROUP, "arcq_act_quant: in_features must be divisible by group_size");
    if (x_dtype != ARCQ_F32 && x_dtype != ARCQ_F16) return fail(ARCQ_ERR_DTYPE, "arcq_act_quant: x must be float32 or float16");
    if (x_hat && x_hat_dtype != ARCQ_F32 && x_hat_dtype != ARCQ_F16)
        return fail(ARCQ_ERR_DTYPE, "arcq_act_quant: x_hat must be float32 or float16");
    if (x_hat && x_hat == x && x_hat_dtype != x_dtype)
        return fail(ARCQ_ERR_DTYPE, "arcq_act_quant: x_hat may alias x only when the dtypes match");
    if (rows * cols == 0) return ARCQ_OK;
    if (!x || !thresholds || !codebook) return fail(ARCQ_ERR_NULL, "arcq_act_quant: x, thresholds and codebook must not be NULL");
    if (rows * (cols / group_size) >= (int64_t(1) << 36)) return fail(ARCQ_ERR_SHAPE, "arcq_act_quant: tensor too large");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int od = x_hat ? x_hat_dtype : x_dtype;
#define ARCQ_GO(TI, TO) \
    return launch<TI, TO>(x, thresholds, codebook, packed, codes_u8, center, scale, code_sum, x_hat, rows, cols, bits, group_size, eps, st)
    if (x_dtype == ARCQ_F32 && od == ARCQ_F32) ARCQ_GO(float, float);
    if (x_dtype == ARCQ_F32 && od == ARCQ_F16) ARCQ_GO(float, __half);
    if (x_dtype == ARCQ_F16 && od == ARCQ_F32) ARCQ_GO(__half, float);
    ARCQ_GO(__half, __half);
#undef ARCQ_GO
}
