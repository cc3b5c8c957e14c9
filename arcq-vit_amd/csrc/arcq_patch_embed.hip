// Front end of a ViT in one launch: the 16 x 16 stride-16 patch convolution as an MFMA product straight from the NCHW
// image (no im2col tensor), its bias, the class token in front and the position embedding added:
//
//   out[b, 0, :]     = cls + pos[0]
//   out[b, 1 + p, :] = fp16( fp16( patch(b, p) . w^T + bias ) + pos[1 + p] ),   p = py * (W / 16) + px
//
// img [B, 3, H, W] fp16, w [N, 3 * 16 * 16] fp16 (a Conv2d weight as it lies: k = c * 256 + i * 16 + j), bias / cls [N],
// pos [1 + (H/16)(W/16), N], out [B, 1 + (H/16)(W/16), N], all fp16.  fp32 accumulation; the two roundings are those of
// the separate convolution and addition it replaces.
//
// No counterpart in the reference's packed path (the fp16 patch embedding of its models is a torch convolution); here
// because with the blocks down to five launches each, torch's im2col + GEMM + concatenation + addition are the largest
// single item of a batch-1 forward.  The quantized patch convolution (ARCQPackedPatchConv) does not go through this.
//
// A k-step of 16 covers half of one 16-pixel image row of a patch: the eight values a lane needs of it are 16
// contiguous bytes of the image, so the fragments are plain 16-byte loads from the image (and from w, whose row is the
// patch in the same order).  Three kernels: patch_embed_kernel (workgroup = 256 patches x 32 channels, weight rows in LDS),
// patch_embed_rows_kernel (many patches, 128 to 384 channels: workgroup = 64 patches x all channels, patches in LDS; patch_rows_pay)
// and, up to 256 tiles of 32 x 32, patch_embed_small_kernel (a workgroup per tile, the k-steps split over its waves).
#include "arcq_common.h"
#include "arcq_gemm.h"

namespace arcq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kPatch = 16, kChannels = 3, kK = kChannels * kPatch * kPatch, kSteps = kK / 16;      // 768, 48

// Workgroup = 256 patches (four waves of 64) x 32 channels.  The 32 weight rows (48 KB) are copied into LDS once, with
// coalesced loads, and every wave reads its weight fragments from there: straight from global memory a weight
// fragment touches 32 different cache lines per instruction (one row each), which costs the vector memory path a clock
// per line and bounded the launch; an image fragment is 1 KB in two or three contiguous runs and stays a global load.
constexpr int kTM = 2;                                  // 32-patch blocks per wave
constexpr int kWPitch = kK * 2 + 16;                    // bytes per weight row in LDS (odd number of 16-byte pieces)

__global__ void __launch_bounds__(256)
patch_embed_kernel(const __half *__restrict__ img, const __half *__restrict__ w, const __half *__restrict__ bias,
                   const __half *__restrict__ cls, const __half *__restrict__ pos, __half *__restrict__ out, int B, int H,
                   int W, int N, int row_groups, int col_tiles)
{
    __shared__ __attribute__((aligned(16))) unsigned char ws[32 * kWPitch];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int pw = W / kPatch, np = (H / kPatch) * pw;
    const int M = B * np;
    const int tiles = row_groups * col_tiles;
    if (static_cast<int>(blockIdx.x) >= tiles) {        // the class-token rows: element e = b * N + n
        const int64_t e0 = (static_cast<int64_t>(blockIdx.x - tiles) * 256 + tid) * 8;
        if (e0 < static_cast<int64_t>(B) * N) {
            const int b = static_cast<int>(e0 / N), n = static_cast<int>(e0 - static_cast<int64_t>(b) * N);
            __half *dst = out + static_cast<int64_t>(b) * (np + 1) * N + n;
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[i] = __float2half_rn(__half2float(cls[n + i]) + __half2float(pos[n + i]));
        }
        return;
    }
    const int rg = blockIdx.x / col_tiles, ct = blockIdx.x - rg * col_tiles;      // neighbours share the patches
    const int n0 = ct * 32;
    // ---- the weight rows n0 .. n0 + 31 into LDS: 3072 pieces of 16 bytes, twelve per thread, all in flight ----
    {
        constexpr int kPiecesPerRow = kK / 8;           // 96
        u32x4_t t[12];
#pragma unroll
        for (int j = 0; j < 12; ++j) {
            const int p = tid + 256 * j, row = p / kPiecesPerRow, col = p - row * kPiecesPerRow;
            t[j] = *reinterpret_cast<const u32x4_t *>(w + static_cast<int64_t>(n0 + row) * kK + col * 8);
        }
#pragma unroll
        for (int j = 0; j < 12; ++j) {
            const int p = tid + 256 * j, row = p / kPiecesPerRow, col = p - row * kPiecesPerRow;
            *reinterpret_cast<u32x4_t *>(ws + row * kWPitch + col * 16) = t[j];
        }
    }
    // per row block: this lane's patch, its first image row (channel 0, i = 0) at column 8 lh, its output row
    const __half *a_base[kTM];
    int64_t out_row[kTM];
    int pos_row[kTM];
    bool valid[kTM];
#pragma unroll
    for (int tm = 0; tm < kTM; ++tm) {
        const int m = ((rg * 4 + wave) * kTM + tm) * 32 + lr;
        const int mc = min(m, M - 1);
        const int b = mc / np, p = mc - b * np, py = p / pw, px = p - py * pw;
        a_base[tm] = img + (static_cast<int64_t>(b) * kChannels * H + py * kPatch) * W + px * kPatch + 8 * lh;
        out_row[tm] = static_cast<int64_t>(b) * (np + 1) + 1 + p;
        pos_row[tm] = 1 + p;
        valid[tm] = m < M;
    }
    const int64_t plane = static_cast<int64_t>(H) * W;
    auto load_step = [&](int s, u32x4_t (&af)[kTM]) {
        const int c = s >> 4, i = s & 15;
        const int64_t a_off = c * plane + static_cast<int64_t>(i) * W;
#pragma unroll
        for (int tm = 0; tm < kTM; ++tm) af[tm] = *reinterpret_cast<const u32x4_t *>(a_base[tm] + a_off);
    };
    float16_t acc[kTM];
#pragma unroll
    for (int tm = 0; tm < kTM; ++tm)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[tm][v] = 0.0f;
    constexpr int kAhead = 8;                  // k-steps of image fragments in flight
    u32x4_t af[kAhead][kTM];
#pragma unroll
    for (int s = 0; s < kAhead - 1; ++s) load_step(s, af[s]);
    __syncthreads();                           // the weight rows are in LDS
    const unsigned char *w_lane = ws + lr * kWPitch + lh * 16;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        if (s + kAhead - 1 < kSteps) load_step(s + kAhead - 1, af[(s + kAhead - 1) % kAhead]);
        const half8_t wb = *reinterpret_cast<const half8_t *>(w_lane + s * 32);
        __builtin_amdgcn_sched_barrier(0);     // (left alone, the compiler sinks the loads towards their use)
#pragma unroll
        for (int tm = 0; tm < kTM; ++tm) {
            half8_t xa;
            __builtin_memcpy(&xa, &af[s % kAhead][tm], 16);
            acc[tm] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb, xa, acc[tm], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // acc[tm][v]: patch lr of row block tm, channel n0 + 8 (v / 4) + 4 lh + v % 4
#pragma unroll
    for (int tm = 0; tm < kTM; ++tm) {
        if (!valid[tm]) continue;
        __half *dst = out + out_row[tm] * N;
        const __half *ps = pos + static_cast<int64_t>(pos_row[tm]) * N;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = n0 + 8 * q + 4 * lh;
            const u32x2_t pv = *reinterpret_cast<const u32x2_t *>(ps + n);
            u32x2_t bv = {0u, 0u};
            if (bias) bv = *reinterpret_cast<const u32x2_t *>(bias + n);
            const __half *ph = reinterpret_cast<const __half *>(&pv), *bh = reinterpret_cast<const __half *>(&bv);
            __half o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const __half y = __float2half_rn(acc[tm][4 * q + e] + __half2float(bh[e]));
                o[e] = __float2half_rn(__half2float(y) + __half2float(ph[e]));
            }
            *reinterpret_cast<u32x2_t *>(dst + n) = *reinterpret_cast<const u32x2_t *>(o);
        }
    }
}

// The same for many patches and 128 to 384 channels: a workgroup owns 64 patches and all channels.  Above, every 32-channel tile reads
// the image again, and 64 images cost 173 MB of traffic for the 29 that they are; here the patches lie in LDS (64 x 768 values, read
// once, in runs of a row's patches), and the weights stream through it 32 values at a time, one barrier a chunk: the next chunk is
// written to the other buffer while later ones are on their way from L2.  Wave = 64 patches x 32 channels (32 x 32 where there are no
// more than six such tiles).  What bounds it is the LDS: 3 KB of reads and 1 of writes for two MFMAs, 15 us for 384 channels however
// few the workgroups; a second pass for more channels loses (768 of 64 images 41 us against 40, of 256 162 / 144).
// 64 images, 384 channels 31.0 -> 21.7 us, 192 channels 24.7 -> 15.8; 256 images 101 -> 90 and 69 -> 63.
constexpr int kRowsWaves = 12, kChunkK = 32, kChunks = kK / kChunkK;      // 24
constexpr int kAPitch = kK * 2 + 16, kBPitch = kChunkK * 2 + 16;          // bytes; odd numbers of 16-byte pieces
constexpr int kRowsN = 32 * kRowsWaves;                                   // the most channels
constexpr int kBBytes = kRowsN * kBPitch;
constexpr int kAheadB = 4;                                                // chunks on their way from L2 or in a buffer
constexpr int kRowsLds = 64 * kAPitch + 2 * kBBytes;

__global__ void __launch_bounds__(64 * kRowsWaves)
patch_embed_rows_kernel(const __half *__restrict__ img, const __half *__restrict__ w, const __half *__restrict__ bias,
                        const __half *__restrict__ cls, const __half *__restrict__ pos, __half *__restrict__ out, int B, int H,
                        int W, int N, int row_tiles)
{
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *as = smem, *bs = smem + 64 * kAPitch;
    constexpr int kThreads = 64 * kRowsWaves;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int pw = W / kPatch, np = (H / kPatch) * pw;
    const int M = B * np;
    if (static_cast<int>(blockIdx.x) >= row_tiles) {        // the class-token rows: element e = b * N + n
        const int64_t e0 = (static_cast<int64_t>(blockIdx.x - row_tiles) * kThreads + tid) * 8;
        if (e0 < static_cast<int64_t>(B) * N) {
            const int b = static_cast<int>(e0 / N), n = static_cast<int>(e0 - static_cast<int64_t>(b) * N);
            __half *dst = out + static_cast<int64_t>(b) * (np + 1) * N + n;
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[i] = __float2half_rn(__half2float(cls[n + i]) + __half2float(pos[n + i]));
        }
        return;
    }
    const int m0 = blockIdx.x * 64;
    // ---- the weights' first four chunks and the patches: 48 image rows x 64 patches x 2 pieces, eight a thread, all in flight.
    // Neighbouring threads take neighbouring patches of one image row. ----
    u32x4_t bt[kAheadB][2];
    auto fetch_b = [&](int c, u32x4_t (&t)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int p = tid + kThreads * j, row = p >> 2, piece = p & 3;
            t[j] = *reinterpret_cast<const u32x4_t *>(w + static_cast<int64_t>(min(row, N - 1)) * kK + c * kChunkK + piece * 8);
        }
    };
    auto store_b = [&](int buf, const u32x4_t (&t)[2]) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int p = tid + kThreads * j;
            *reinterpret_cast<u32x4_t *>(bs + buf * kBBytes + (p >> 2) * kBPitch + (p & 3) * 16) = t[j];
        }
    };
#pragma unroll
    for (int c = 0; c < kAheadB; ++c) fetch_b(c, bt[c]);
    {
        const int pl = (tid >> 1) & 63, h = tid & 1;
        const int mc = min(m0 + pl, M - 1), b = mc / np, p = mc - b * np, py = p / pw, px = p - py * pw;
        const __half *src = img + (static_cast<int64_t>(b) * kChannels * H + py * kPatch) * W + px * kPatch + h * 8;
        u32x4_t at[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int ci = (tid >> 7) + 6 * j, c = ci >> 4, i = ci & 15;      // 768 threads: six image rows a round
            at[j] = *reinterpret_cast<const u32x4_t *>(src + (static_cast<int64_t>(c) * H + i) * W);
        }
        store_b(0, bt[0]);
#pragma unroll
        for (int j = 0; j < 8; ++j) *reinterpret_cast<u32x4_t *>(as + pl * kAPitch + ((tid >> 7) + 6 * j) * 32 + h * 16) = at[j];
    }
    int64_t out_row[2];
    int pos_row[2];
    bool valid[2];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm) {
        const int m = m0 + tm * 32 + lr, mc = min(m, M - 1), b = mc / np, p = mc - b * np;
        out_row[tm] = static_cast<int64_t>(b) * (np + 1) + 1 + p;
        pos_row[tm] = 1 + p;
        valid[tm] = m < M;
    }
    const unsigned char *a_lane = as + lr * kAPitch + lh * 16;
    const int tiles = N / 32;
    const bool halves = tiles <= kRowsWaves / 2;             // two waves a tile, a row block each
    const int ct = halves ? wave % (kRowsWaves / 2) : wave, tm0 = halves ? wave / (kRowsWaves / 2) : 0;
    float16_t acc[2];
#pragma unroll
    for (int tm = 0; tm < 2; ++tm)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[tm][v] = 0.0f;
    const unsigned char *b_lane = bs + (ct * 32 + lr) * kBPitch + lh * 16;
#pragma unroll 4
    for (int c = 0; c < kChunks; ++c) {
        __syncthreads();                                     // chunk c is in buffer c & 1, chunk c - 1 has been read
        store_b((c + 1) & 1, bt[(c + 1) % kAheadB]);
        fetch_b(min(c + kAheadB, kChunks - 1), bt[c % kAheadB]);
#pragma unroll
        for (int s = 0; s < kChunkK / 16; ++s) {
            const half8_t wb = *reinterpret_cast<const half8_t *>(b_lane + (c & 1) * kBBytes + s * 32);
            const half8_t x0 = *reinterpret_cast<const half8_t *>(a_lane + tm0 * 32 * kAPitch + (c * 2 + s) * 32);
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb, x0, acc[0], 0, 0, 0);
            if (!halves) {
                const half8_t x1 = *reinterpret_cast<const half8_t *>(a_lane + 32 * kAPitch + (c * 2 + s) * 32);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb, x1, acc[1], 0, 0, 0);
            }
        }
    }
    // acc[tm][v]: patch lr of row block tm, channel 8 (v / 4) + 4 lh + v % 4 of the tile
    if (ct >= tiles) return;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (i == 1 && halves) break;
        const int tm = halves ? tm0 : i;
        if (!(tm ? valid[1] : valid[0])) continue;
        __half *dst = out + (tm ? out_row[1] : out_row[0]) * N;
        const __half *ps = pos + static_cast<int64_t>(tm ? pos_row[1] : pos_row[0]) * N;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int n = ct * 32 + 8 * q + 4 * lh;
            const u32x2_t pv = *reinterpret_cast<const u32x2_t *>(ps + n);
            u32x2_t bv = {0u, 0u};
            if (bias) bv = *reinterpret_cast<const u32x2_t *>(bias + n);
            const __half *ph = reinterpret_cast<const __half *>(&pv), *bh = reinterpret_cast<const __half *>(&bv);
            __half o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const __half y = __float2half_rn(acc[i][4 * q + e] + __half2float(bh[e]));
                o[e] = __float2half_rn(__half2float(y) + __half2float(ph[e]));
            }
            *reinterpret_cast<u32x2_t *>(dst + n) = *reinterpret_cast<const u32x2_t *>(o);
        }
    }
}

// The same for few patches (batch 1-2): one 32 x 32 tile per workgroup, its 48 k-steps dealt to the four waves (twelve
// each, all 24 fragment loads of a wave in flight at once: the launch is one memory latency, twelve MFMAs and a
// reduction of the four partial tiles through LDS, in wave order).
__global__ void __launch_bounds__(256)
patch_embed_small_kernel(const __half *__restrict__ img, const __half *__restrict__ w, const __half *__restrict__ bias,
                         const __half *__restrict__ cls, const __half *__restrict__ pos, __half *__restrict__ out, int B,
                         int H, int W, int N, int row_tiles, int col_tiles)
{
    __shared__ float part[3][16][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int pw = W / kPatch, np = (H / kPatch) * pw;
    const int M = B * np;
    const int tile = blockIdx.x, tiles = row_tiles * col_tiles;
    if (tile >= tiles) {        // the class-token rows: element e = b * N + n
        const int64_t e0 = (static_cast<int64_t>(tile - tiles) * 256 + tid) * 8;
        if (e0 < static_cast<int64_t>(B) * N) {
            const int b = static_cast<int>(e0 / N), n = static_cast<int>(e0 - static_cast<int64_t>(b) * N);
            __half *dst = out + static_cast<int64_t>(b) * (np + 1) * N + n;
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[i] = __float2half_rn(__half2float(cls[n + i]) + __half2float(pos[n + i]));
        }
        return;
    }
    const int rt = tile / col_tiles, ct = tile - rt * col_tiles;
    const int m = rt * 32 + lr, mc = min(m, M - 1);
    const int b = mc / np, p = mc - b * np, py = p / pw, px = p - py * pw;
    const __half *a_base = img + (static_cast<int64_t>(b) * kChannels * H + py * kPatch) * W + px * kPatch + 8 * lh;
    const __half *w_base = w + static_cast<int64_t>(min(ct * 32 + lr, N - 1)) * kK + 8 * lh;
    const int64_t plane = static_cast<int64_t>(H) * W;
    constexpr int kMine = kSteps / 4;          // 12 k-steps per wave
    u32x4_t af[kMine], bf[kMine];
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
        const int s = wave * kMine + j, c = s >> 4, i = s & 15;
        af[j] = *reinterpret_cast<const u32x4_t *>(a_base + c * plane + static_cast<int64_t>(i) * W);
        bf[j] = *reinterpret_cast<const u32x4_t *>(w_base + s * 16);
    }
    __builtin_amdgcn_sched_barrier(0);         // every load is issued before the first wait
    float16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
        half8_t xa, wb;
        __builtin_memcpy(&xa, &af[j], 16);
        __builtin_memcpy(&wb, &bf[j], 16);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(wb, xa, acc, 0, 0, 0);
    }
    if (wave > 0) {
#pragma unroll
        for (int v = 0; v < 16; ++v) part[wave - 1][v][lane] = acc[v];
    }
    __syncthreads();
    if (wave > 0 || m >= M) return;
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] += part[q][v][lane];
    __half *dst = out + (static_cast<int64_t>(b) * (np + 1) + 1 + p) * N;
    const __half *ps = pos + static_cast<int64_t>(1 + p) * N;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = ct * 32 + 8 * q + 4 * lh;
        const u32x2_t pv = *reinterpret_cast<const u32x2_t *>(ps + n);
        u32x2_t bv = {0u, 0u};
        if (bias) bv = *reinterpret_cast<const u32x2_t *>(bias + n);
        const __half *ph = reinterpret_cast<const __half *>(&pv), *bh = reinterpret_cast<const __half *>(&bv);
        __half o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const __half y = __float2half_rn(acc[4 * q + e] + __half2float(bh[e]));
            o[e] = __float2half_rn(__half2float(y) + __half2float(ph[e]));
        }
        *reinterpret_cast<u32x2_t *>(dst + n) = *reinterpret_cast<const u32x2_t *>(o);
    }
}

// Where patch_embed_rows_kernel is the faster one.  Its workgroups have a compute unit each, so it takes whole rounds of them, about
// 2 N / 32 + 3 parts a round (the channels, the patches); the other kernel's (256 patches x 32 channels) are a sixth to a fifth of a
// round and several share a compute unit.  Measured at 160 to 1 500 tiles of 64 patches, 224 x 224 and 128 x 128 images, us here / there:
//   one round      384 channels, 160 tiles 20.4 / 23.5, 224 22.7 / 32.2; 192: 14.9 / 17.6, 15.7 / 25.7; 128: 13.6 / 13.1, 14.5 / 16.8;
//                  96: 12.9 / 11.2, 13.6 / 13.6; fewer tiles: 384 channels, 98 tiles 20.1 / 20.4, 192 15.4 / 12.7
//   a second begun 257 tiles: 384 channels 39.1 / 37.2, 320 36.8 / 34.3, 256 33.8 / 35.8, 224 31.6 / 28.4, 192 28.1 / 25.9, 160 26.4 / 24.2;
//                  304: 42.1 / 42.1, 38.6 / 39.0, 35.4 / 40.0, 32.9 / 38.5, 29.9 / 29.3, 27.9 / 26.2; 350: 42.8 / 50.7, 39.2 / 47.0,
//                  35.8 / 42.6, 33.3 / 40.0, 30.4 / 38.9, 28.6 / 28.3; 512: 52.5 / 65.1, 192 channels 36.7 / 46.3
//   more           513: 63.7 / 66.0, 192 channels 45.7 / 49.4, 160 42.6 / 39.6; 784: 90.5 / 101, 63.2 / 69.3, 59.0 / 58.4
bool patch_rows_pay(int64_t M, int64_t n)
{
    const int64_t cus = device_cus(), tiles = (M + 63) / 64;
    if (n < 128 || n > kRowsN || tiles * 16 < cus * (n < 160 ? 11 : 10)) return false;
    const int64_t rounds = (tiles + cus - 1) / cus;
    if (rounds == 1) return true;
    const int64_t groups = (M + 128 * kTM - 1) / (128 * kTM), others = (groups * (n / 32) + cus - 1) / cus;      // the other kernel's on a compute unit
    return n >= 160 && 5 * rounds * (2 * (n / 32) + 3) <= 64 * others;
}

}  // namespace
}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_patch_embed_fwd(const void *img, const void *w, const void *bias, const void *cls, const void *pos, void *out,
                                  int64_t B, int64_t H, int64_t W, int64_t patch, int64_t N, void *stream)
{
    if (B < 0 || H < 0 || W < 0 || N < 0) return fail(ARCQ_ERR_SHAPE, "arcq_patch_embed_fwd: negative size");
    if (patch != kPatch) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_patch_embed_fwd: patch size must be 16 (got %lld)", static_cast<long long>(patch));
    if (H % kPatch || W % kPatch) return fail(ARCQ_ERR_SHAPE, "arcq_patch_embed_fwd: image sides must be multiples of 16");
    if (N % 32) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_patch_embed_fwd: embedding width must be a multiple of 32 (got %lld)", static_cast<long long>(N));
    if (B == 0 || N == 0) return ARCQ_OK;
    if (H == 0 || W == 0) return fail(ARCQ_ERR_SHAPE, "arcq_patch_embed_fwd: empty image");
    if (!img || !w || !cls || !pos || !out) return fail(ARCQ_ERR_NULL, "arcq_patch_embed_fwd: NULL tensor pointer");
    if (!aligned(img, 16) || !aligned(w, 16) || !aligned(out, 8) || !aligned(pos, 8) || (bias && !aligned(bias, 8)))
        return fail(ARCQ_ERR_ALIGN, "arcq_patch_embed_fwd: img and w must be 16-byte, bias / pos / out 8-byte aligned");
    const int64_t M = B * (H / kPatch) * (W / kPatch);
    if (B > (1 << 20) || H > (1 << 14) || W > (1 << 14) || N > (1 << 16) || M >= (int64_t(1) << 30) || (M + B) * N >= (int64_t(1) << 40))
        return fail(ARCQ_ERR_SHAPE, "arcq_patch_embed_fwd: tensor too large");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int b = static_cast<int>(B), h = static_cast<int>(H), wd = static_cast<int>(W), n = static_cast<int>(N);
    const auto *pi = static_cast<const __half *>(img), *pwt = static_cast<const __half *>(w), *pb = static_cast<const __half *>(bias);
    const auto *pc = static_cast<const __half *>(cls), *pp = static_cast<const __half *>(pos);
    auto *po = static_cast<__half *>(out);
    const int cls_wgs = static_cast<int>((B * N / 8 + 255) / 256);
    const int col_tiles = n / 32;
    if (((M + 31) / 32) * col_tiles <= 256) {
        const int row_tiles = static_cast<int>((M + 31) / 32);
        hipLaunchKernelGGL(patch_embed_small_kernel, dim3(row_tiles * col_tiles + cls_wgs), dim3(256), 0, st, pi, pwt, pb, pc, pp, po,
                           b, h, wd, n, row_tiles, col_tiles);
    } else if (patch_rows_pay(M, n)) {
        allow_dynamic_lds<patch_embed_rows_kernel>(kRowsLds);
        const int row_tiles = static_cast<int>((M + 63) / 64);
        hipLaunchKernelGGL(patch_embed_rows_kernel, dim3(row_tiles + (cls_wgs + 2) / 3), dim3(64 * kRowsWaves), kRowsLds, st, pi, pwt, pb, pc, pp, po,
                           b, h, wd, n, row_tiles);
    } else {
        const int row_groups = static_cast<int>((M + 128 * kTM - 1) / (128 * kTM));      // four waves of 32 kTM patches
        hipLaunchKernelGGL(patch_embed_kernel, dim3(row_groups * col_tiles + cls_wgs), dim3(256), 0, st, pi, pwt, pb, pc, pp, po, b, h, wd,
                           n, row_groups, col_tiles);
    }
    return launch_status("arcq_patch_embed_fwd");
}
