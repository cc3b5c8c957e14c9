// Stage 3 on prepared operands: y[M,N] = x_hat[M,K] * w_hat[N,K]^T + bias with both operands fp16 in the 32-row block
// layout (x_hat [M/32][K/8][32 rows][8], a last block of r < 32 rows stored compactly; w_hat [N/32][K/8][32 columns][8],
// N a multiple of 32), as arcq_prepare writes them.  For the shapes between "a few hundred rows" and "enough row blocks
// for the weight-stationary kernels" -- most batches of a ViT -- where those kernels leave most of the chip idle: a
// 128-column slab per workgroup is 8 slabs x 19 row blocks at 591 x 1024, one or two of a workgroup's eight waves multiply
// at a time, and the chain over K = 4096 took 34 us.
//
// gemm_tile_kernel (M >= 512): TM x TN output tiles, every wave a fixed part of the tile for all of K (ascending k, so the
// bits are those of the other large-M kernels).  Both operands are staged group by group (64 k-values: 4 KB per 32-row
// block, contiguous in the block layout) by direct global -> LDS loads, kStages - 1 groups ahead, one barrier per group;
// a fragment is one conflict-free 16-byte LDS read.  Bound by the L1 / LDS streams of (TM + TN) * 128 bytes per group at
// the small tiles (256 clocks per group and workgroup for 64 x 64, MFMA 128), by both and the MFMAs at 128 x 128.
//
// gemm_tile_split_kernel (M < 512): 32- or 64-row tiles, K split over eight waves exactly as gemm_splitk_kernel splits it
// (wave w: groups w, w + 8, ...; partial tiles added in LDS in the order 0 .. 7, then the bias): the same bits, without
// rebuilding the weights in every row tile.  Fragments go straight from L2 to registers (512 contiguous bytes per half wave).
//
// k order inside a group: lane half h covers k = 32 h + 8 step ... + 7 in k-step `step`.  w_hat is the MFMA "A" operand:
// accumulator element v of lane l is y[m = 32 i + l % 32][n = 32 j + 8 (v / 4) + 4 (l / 32) + v % 4].
#include "arcq_act_quant_core.h"
#include "arcq_gemm.h"

#include <algorithm>
#include <type_traits>

namespace arcq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kStages = 4;
constexpr int kGroupBytes = 4096;           // 32 rows x 64 values (FP8: 128 values)

template <int V> __device__ __forceinline__ void wait_vm()
{
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(V) : "memory");
}

// FP8 operands: one MFMA of 64 k-values from two 16-byte pieces of each operand.
__device__ __forceinline__ float16_t mfma_fp8(const u32x4_t (&w)[2], const u32x4_t (&x)[2], const float16_t &acc)
{
    i32x8_t wf, xf;
    __builtin_memcpy(&wf, &w, 32);
    __builtin_memcpy(&xf, &x, 32);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf, xf, acc, 0, 0, 0, 0, 0, 0);
}

// Outputs of an accumulator register block -> fp16 / fp32 in an LDS tile (rows `pitch` bytes apart), bias added (F8: after the
// multiplication by `inv`, a power of two, which is exact).
template <typename TOUT, bool F8>
__device__ __forceinline__ void stage_block(const float16_t &acc, const float *s_bias, unsigned char *tile, int pitch, int lr, int lh,
                                            float inv)
{
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 b = *reinterpret_cast<const float4 *>(s_bias + 8 * q + 4 * lh);
        float a[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = F8 ? acc[4 * q + e] * inv : acc[4 * q + e];
        const float o0 = a[0] + b.x, o1 = a[1] + b.y, o2 = a[2] + b.z, o3 = a[3] + b.w;
        unsigned char *dst = tile + lr * pitch + (8 * q + 4 * lh) * static_cast<int>(sizeof(TOUT));
        if constexpr (sizeof(TOUT) == 2) {
            const __half2 lo = __floats2half2_rn(o0, o1), hi = __floats2half2_rn(o2, o3);
            u32x2_t pk;
            pk[0] = *reinterpret_cast<const uint32_t *>(&lo);
            pk[1] = *reinterpret_cast<const uint32_t *>(&hi);
            *reinterpret_cast<u32x2_t *>(dst) = pk;
        } else {
            u32x4_t pk;
            pk[0] = __float_as_uint(o0); pk[1] = __float_as_uint(o1);
            pk[2] = __float_as_uint(o2); pk[3] = __float_as_uint(o3);
            *reinterpret_cast<u32x4_t *>(dst) = pk;
        }
    }
}

// WM x WN waves per workgroup; NQ = 0 or the bits of the consuming layer's quantizer (y then receives its x_hat).
template <int TM, int TN, int WM, int WN, typename TOUT, int NQ, bool F8>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_tile_kernel(const unsigned char *__restrict__ xb, const unsigned char *__restrict__ wb, const float *__restrict__ bias,
                 TOUT *__restrict__ y, int M, int N, int G, int m_tiles, int n_tiles, int m_fastest,
                 const TOUT *__restrict__ residual, int gelu, const float *__restrict__ nx_thr, const float *__restrict__ nx_cb, float inv)
{
    constexpr int kWaves = WM * WN, kThreads = 64 * kWaves;
    constexpr int RBT = TM / 32, CBT = TN / 32;                  // 32-row / 32-column blocks of the tile
    constexpr int RB = RBT / WM, CB = CBT / WN;                  // of a wave
    constexpr int kStageBytes = (RBT + CBT) * kGroupBytes;
    constexpr int LPW = (RBT + CBT) * 4 / kWaves;                // 1 KB loads per wave and group
    static_assert((RBT + CBT) * 4 % kWaves == 0, "loads must deal evenly: the waits count them");
    constexpr int kOutPitch = TN * static_cast<int>(sizeof(TOUT)) + 16;
    static_assert(TM * kOutPitch <= kStages * kStageBytes, "the output tile reuses the operand stages");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    float *s_bias = reinterpret_cast<float *>(smem + kStages * kStageBytes);      // [TN]
    unsigned char *nq_lds = reinterpret_cast<unsigned char *>(s_bias + TN);

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, lh = lane >> 5;
    // Tiles are dealt so that each XCD takes a contiguous run; along the run the operand that is cheaper to fetch once
    // per XCD is the one that repeats (m_fastest: few rows, every XCD reads all of x_hat and an eighth of the weights).
    const int tiles = m_tiles * n_tiles;
    const int per_xcd = (tiles + 7) / 8;
    const int tile_no = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per_xcd || tile_no >= tiles) return;
    const int mt = m_fastest ? tile_no % m_tiles : tile_no / n_tiles;
    const int nt = m_fastest ? tile_no / m_tiles : tile_no % n_tiles;
    const int m0 = mt * TM, n0 = nt * TN;
    const int row_blocks = (M + 31) / 32, col_blocks = N / 32;

    // This wave's loads: load q moves the quarter q % 4 of block q / 4 of the stage.  LDS always holds 32 rows per piece
    // column; for a compact last block of r rows lane (k8, row) reads row min(row, r - 1), so every lane's address is
    // inside the tensor and every wave issues the same number of loads per group (the waits below count them).
    const char *src[LPW];
    uint32_t voff[LPW], gstep[LPW];
#pragma unroll
    for (int j = 0; j < LPW; ++j) {
        const int q = wave * LPW + j, b = q >> 2, quarter = q & 3;
        const int piece = quarter * 64 + lane;                       // k8 * 32 + row
        if (b < RBT) {
            const int blk = min(m0 / 32 + b, row_blocks - 1);
            const int r = min(32, M - blk * 32);
            src[j] = reinterpret_cast<const char *>(xb) + static_cast<int64_t>(blk) * G * kGroupBytes;
            voff[j] = static_cast<uint32_t>(((piece >> 5) * r + min(piece & 31, r - 1)) * 16);
            gstep[j] = static_cast<uint32_t>(r * 128);
        } else {
            const int blk = min(n0 / 32 + (b - RBT), col_blocks - 1);
            src[j] = reinterpret_cast<const char *>(wb) + static_cast<int64_t>(blk) * G * kGroupBytes;
            voff[j] = static_cast<uint32_t>(piece * 16);
            gstep[j] = kGroupBytes;
        }
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) unsigned char *)(smem + wave * LPW * 1024))));
    auto issue = [&](int slot) __attribute__((always_inline)) {        // the next group in order into stage `slot`
#pragma unroll
        for (int j = 0; j < LPW; ++j) {
            const uint32_t lds = lds0 + static_cast<uint32_t>(slot * kStageBytes + j * 1024);
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff[j]), "s"(src[j]), "s"(lds) : "memory", "m0");
            src[j] += gstep[j];
        }
    };
    for (int i = tid; i < TN; i += kThreads) s_bias[i] = (bias && n0 + i < N) ? bias[n0 + i] : 0.0f;
    if constexpr (NQ != 0) {
        if (wave == 0) next_quant_setup<NQ>(load_quant_params<NQ>(nx_thr, nx_cb, lane), nq_lds, lane);
    }
    wait_vm<0>();          // nothing but the operand loads is outstanding from here to the epilogue
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
        if (s < G) issue(s);

    float16_t acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    const int wm = wave / WN, wn = wave - wm * WN;
    constexpr int kHalf = F8 ? 1024 : 2048;      // FP8: lane half h covers k = 64 step + 32 h ... + 31, two pieces
    const unsigned char *a_lane = smem + wm * RB * kGroupBytes + lh * kHalf + lr * 16;
    const unsigned char *b_lane = smem + (RBT + wn * CB) * kGroupBytes + lh * kHalf + lr * 16;
    for (int g = 0; g < G; ++g) {
        // Group g has landed for this wave; after the barrier for all of them, and everyone is done with group g - 1.
        const int ahead = G - 1 - g;
        if (ahead >= kStages - 2) wait_vm<(kStages - 2) * LPW>();
        else if (ahead == 1) wait_vm<LPW>();
        else wait_vm<0>();
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (g + kStages - 1 < G) issue((g + kStages - 1) % kStages);
        const int off = (g % kStages) * kStageBytes;
        if constexpr (F8) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                u32x4_t af[RB][2], bf[CB][2];
#pragma unroll
                for (int p = 0; p < 2; ++p) {
#pragma unroll
                    for (int i = 0; i < RB; ++i) af[i][p] = *reinterpret_cast<const u32x4_t *>(a_lane + off + i * kGroupBytes + s * 2048 + p * 512);
#pragma unroll
                    for (int j = 0; j < CB; ++j) bf[j][p] = *reinterpret_cast<const u32x4_t *>(b_lane + off + j * kGroupBytes + s * 2048 + p * 512);
                }
#pragma unroll
                for (int i = 0; i < RB; ++i)
#pragma unroll
                    for (int j = 0; j < CB; ++j) acc[i][j] = mfma_fp8(bf[j], af[i], acc[i][j]);
            }
        } else
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            half8_t af[RB], bf[CB];
#pragma unroll
            for (int i = 0; i < RB; ++i) af[i] = *reinterpret_cast<const half8_t *>(a_lane + off + i * kGroupBytes + kk * 512);
#pragma unroll
            for (int j = 0; j < CB; ++j) bf[j] = *reinterpret_cast<const half8_t *>(b_lane + off + j * kGroupBytes + kk * 512);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
    }
    static_assert(kStages == 4, "the tail waits above assume four stages");

    // ---- epilogue: the tile through LDS, then whole rows of it in 16-byte pieces ----
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
            stage_block<TOUT, F8>(acc[i][j], s_bias + (wn * CB + j) * 32, smem + (wm * RB + i) * 32 * kOutPitch + (wn * CB + j) * 32 * static_cast<int>(sizeof(TOUT)),
                                  kOutPitch, lr, lh, inv);
    __syncthreads();
    if constexpr (NQ != 0) {
        static_assert(TN % 64 == 0 && sizeof(TOUT) == 2, "whole groups of fp16 outputs");
        constexpr int kJobs = RBT * (TN / 64);
        for (int job = wave; job < kJobs; job += kWaves) {
            const int rb = job % RBT, gc = job / RBT;
            const int blk = m0 / 32 + rb, c0 = n0 + gc * 64;
            if (blk < row_blocks && c0 < N)
                next_quant_block<NQ, F8>(nq_lds, smem + rb * 32 * kOutPitch + gc * 128, kOutPitch, lane, gelu != 0, 1.0e-6f, y, blk, M,
                                         N, c0);
        }
    } else {
        constexpr int kVec = 16 / static_cast<int>(sizeof(TOUT));
        constexpr int kPieces = TN / kVec;                        // per row
        constexpr int kRounds = TM * kPieces / kThreads;
#pragma unroll 4
        for (int i = 0; i < kRounds; ++i) {
            const int p = i * kThreads + tid;
            const int r = p / kPieces, c = p % kPieces;
            const int row = m0 + r, col = n0 + c * kVec;
            if (row < M && col < N) {                             // (N is a multiple of 32: whole pieces)
                u32x4_t v = *reinterpret_cast<const u32x4_t *>(smem + r * kOutPitch + c * 16);
                const int64_t at = static_cast<int64_t>(row) * N + col;
                if (residual || gelu) post_ops16<TOUT>(v, residual ? residual + at : nullptr, gelu != 0, kVec);
                store_streaming16(y + at, v[0], v[1], v[2], v[3]);
            }
        }
    }
}

template <int TM, int TN, int WM, int WN, typename TOUT, int NQ, bool F8>
void launch_tile(const GemmArgs &g, const void *w_hat, hipStream_t stream)
{
    constexpr int kSmem = kStages * (TM / 32 + TN / 32) * kGroupBytes + TN * 4 + (NQ ? next_quant_lds_bytes() : 0);
    allow_dynamic_lds<gemm_tile_kernel<TM, TN, WM, WN, TOUT, NQ, F8>>(kSmem);
    const int mt = (g.M + TM - 1) / TM, nt = (g.N + TN - 1) / TN;
    const int m_fastest = g.M < g.N ? 1 : 0;
    hipLaunchKernelGGL((gemm_tile_kernel<TM, TN, WM, WN, TOUT, NQ, F8>), dim3(8 * ((mt * nt + 7) / 8)), dim3(64 * WM * WN), kSmem, stream,
                       static_cast<const unsigned char *>(g.x_hat), static_cast<const unsigned char *>(w_hat), g.bias,
                       static_cast<TOUT *>(g.y), g.M, g.N, operand_units(g.K, F8), mt, nt, m_fastest, static_cast<const TOUT *>(g.residual),
                       g.gelu ? 1 : 0, g.next_thr, g.next_cb, g.fp8_inv);
}

// ---- fewer than 512 rows ------------------------------------------------------------------------------------------
template <typename TOUT, int RB, int CB, int NQ>
__global__ void __launch_bounds__(512)
gemm_tile_split_kernel(const unsigned char *__restrict__ xb, const unsigned char *__restrict__ wb, const float *__restrict__ bias,
                       TOUT *__restrict__ y, int M, int N, int G, const TOUT *__restrict__ residual, int gelu,
                       const float *__restrict__ nx_thr, const float *__restrict__ nx_cb)
{
    constexpr int NW = 8;
    constexpr int RT = 32 * RB, CT = 32 * CB;
    constexpr int kPitch = CT * 4 + 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];      // [NW][RT][kPitch] partial tiles
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int m0 = blockIdx.y * RT, n0 = blockIdx.x * CT;
    const int row_blocks = (M + 31) / 32, col_blocks = N / 32;
    const char *a_src[RB], *b_src[CB];
    int a_step[RB];                      // bytes between k-steps
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int blk = min(m0 / 32 + i, row_blocks - 1);
        const int r = min(32, M - blk * 32);
        a_step[i] = r * 16;
        a_src[i] = reinterpret_cast<const char *>(xb) + static_cast<int64_t>(blk) * G * kGroupBytes + lh * 4 * a_step[i] + min(lr, r - 1) * 16;
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int blk = min(n0 / 32 + j, col_blocks - 1);
        b_src[j] = reinterpret_cast<const char *>(wb) + static_cast<int64_t>(blk) * G * kGroupBytes + lh * 2048 + lr * 16;
    }
    struct Ops { u32x4_t a[RB][4], b[CB][4]; };
    auto fetch = [&](int g, Ops &o) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
            for (int i = 0; i < RB; ++i) o.a[i][kk] = *reinterpret_cast<const u32x4_t *>(a_src[i] + (g * 8 + kk) * a_step[i]);
#pragma unroll
            for (int j = 0; j < CB; ++j) o.b[j][kk] = *reinterpret_cast<const u32x4_t *>(b_src[j] + g * kGroupBytes + kk * 512);
        }
    };
    Ops o0, o1;
    QuantParams nq_params{};
    if constexpr (NQ != 0) {                                          // (the last wave: without operands of its own up to seven groups)
        if (wave == NW - 1) nq_params = load_quant_params<NQ>(nx_thr, nx_cb, lane);
    }
    if (wave < G) fetch(wave, o0);
    if (wave + NW < G) fetch(wave + NW, o1);
    // The consumer's lookup tables while the first operands are on their way.
    unsigned char *nq_lds = smem + NW * RT * kPitch;
    if constexpr (NQ != 0) {
        if (wave == NW - 1) next_quant_setup<NQ>(nq_params, nq_lds, lane);
    }

    float16_t acc[RB][CB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    auto compute = [&](const Ops &o) __attribute__((always_inline)) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            half8_t af[RB], bf[CB];
#pragma unroll
            for (int i = 0; i < RB; ++i) __builtin_memcpy(&af[i], &o.a[i][kk], 16);
#pragma unroll
            for (int j = 0; j < CB; ++j) __builtin_memcpy(&bf[j], &o.b[j][kk], 16);
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int j = 0; j < CB; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
    };
    // The thread's outputs in the epilogue: bias and residual are requested here, under the product.
    constexpr int E = RT * CT / (NW * 64);                     // consecutive outputs per thread (8, 4 or 2)
    constexpr int TPR = CT / E;
    constexpr int BYTES = E * static_cast<int>(sizeof(TOUT));
    const int row = tid / TPR, col = (tid % TPR) * E;
    const int gr = m0 + row, gc = n0 + col;
    const bool live = gr < M && gc < N;                        // (N a multiple of 32: all E outputs or none)
    float bv[E];
    TOUT rv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) bv[e] = 0.0f, rv[e] = from_float<TOUT>(0.0f);
    if (live) {
        if (bias) {
#pragma unroll
            for (int e = 0; e < E; ++e) bv[e] = bias[gc + e];
        }
        if (residual) __builtin_memcpy(rv, __builtin_assume_aligned(residual + static_cast<int64_t>(gr) * N + gc, BYTES < 16 ? BYTES : 16), BYTES);
    }
    for (int g = wave; g < G; g += 2 * NW) {
        compute(o0);
        if (g + 2 * NW < G) fetch(g + 2 * NW, o0);
        if (g + NW < G) {
            compute(o1);
            if (g + 3 * NW < G) fetch(g + 3 * NW, o1);
        }
    }
    unsigned char *mine = smem + wave * (RT * kPitch);
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4_t v;
                v[0] = acc[i][j][4 * q]; v[1] = acc[i][j][4 * q + 1]; v[2] = acc[i][j][4 * q + 2]; v[3] = acc[i][j][4 * q + 3];
                *reinterpret_cast<f32x4_t *>(mine + (i * 32 + lr) * kPitch + (j * 32 + 8 * q + 4 * lh) * 4) = v;
            }
    __syncthreads();
    float sum[E];
#pragma unroll
    for (int e = 0; e < E; ++e) sum[e] = 0.0f;
    const int used = min(NW, G);                               // the other waves hold zeros
    for (int w = 0; w < used; ++w) {
        const unsigned char *src = smem + w * (RT * kPitch) + row * kPitch + col * 4;
        if constexpr (E % 4 == 0) {
#pragma unroll
            for (int e = 0; e < E; e += 4) {
                const f32x4_t v = *reinterpret_cast<const f32x4_t *>(src + e * 4);
                sum[e] += v[0]; sum[e + 1] += v[1]; sum[e + 2] += v[2]; sum[e + 3] += v[3];
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) sum[e] += *reinterpret_cast<const float *>(src + e * 4);
        }
    }
    TOUT out[E];
#pragma unroll
    for (int e = 0; e < E; ++e) out[e] = from_float<TOUT>(sum[e] + bv[e]);
    if constexpr (NQ != 0) {
        // A row's 64 columns are a group of the consumer, which its TPR neighbouring lanes hold: stage 1 in their registers, on all
        // waves.  (As an fp16 tile in LDS that one wave per 32 rows quantized, two lanes a group: 384 -> 1 536 at 197 rows 6.0 us, now 5.2;
        // 1 024 -> 4 096 10.0 -> 9.4.)
        static_assert(CT == 64 && sizeof(TOUT) == 2 && (E == 4 || E == 8), "whole groups of fp16 outputs");
        float v[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (gelu) out[e] = post_op1<TOUT>(out[e], false, rv[e], true);
            v[e] = to_float(out[e]);
        }
        next_quant_lanes<NQ>(nq_lds, v, lane, 1.0e-6f);
        uint32_t o[4];
#pragma unroll
        for (int d = 0; d < E / 2; ++d) {
            const __half2 h = __floats2half2_rn(v[2 * d], v[2 * d + 1]);
            o[d] = *reinterpret_cast<const uint32_t *>(&h);
        }
        if constexpr (E == 4) {      // (the even lane stores its neighbour's half of the 16-byte piece)
            o[2] = __float_as_uint(from_odd_lane(__uint_as_float(o[0])));
            o[3] = __float_as_uint(from_odd_lane(__uint_as_float(o[1])));
        }
        if (live && (E == 8 || !(lane & 1))) {
            const int blk = gr >> 5, rows = min(32, M - blk * 32);
            store_writethrough16(reinterpret_cast<char *>(y) + static_cast<int64_t>(blk) * 64 * N + (static_cast<int64_t>(gc / 8) * rows + (gr & 31)) * 16,
                                 o[0], o[1], o[2], o[3]);
        }
    } else if (live) {
        if (residual || gelu) {
#pragma unroll
            for (int e = 0; e < E; ++e) out[e] = post_op1<TOUT>(out[e], residual != nullptr, rv[e], gelu != 0);
        }
        TOUT *dst = y + static_cast<int64_t>(gr) * N + gc;
        __builtin_memcpy(__builtin_assume_aligned(dst, BYTES < 16 ? BYTES : 16), out, BYTES);
    }
}

template <typename TOUT, int RB, int CB, int NQ>
void launch_split(const GemmArgs &g, const void *w_hat, hipStream_t stream)
{
    constexpr int kSmem = 8 * 32 * RB * (32 * CB * 4 + 16) + (NQ ? next_quant_lds_bytes() : 0);
    allow_dynamic_lds<gemm_tile_split_kernel<TOUT, RB, CB, NQ>>(kSmem);
    const dim3 grid((g.N + 32 * CB - 1) / (32 * CB), (g.M + 32 * RB - 1) / (32 * RB));
    hipLaunchKernelGGL((gemm_tile_split_kernel<TOUT, RB, CB, NQ>), grid, dim3(512), kSmem, stream,
                       static_cast<const unsigned char *>(g.x_hat), static_cast<const unsigned char *>(w_hat), g.bias,
                       static_cast<TOUT *>(g.y), g.M, g.N, g.K / 64, static_cast<const TOUT *>(g.residual), g.gelu ? 1 : 0, g.next_thr,
                       g.next_cb);
}

template <typename TOUT, int NQ, bool F8>
void pick(const GemmArgs &g, const void *w_hat, hipStream_t stream)
{
    const int cus = device_cus();
    if (!F8 && g.M < 512) {      // (FP8: one order of k at every M, the order of the other FP8 kernel)
        // The smallest tile whose launch is one round of workgroups (one per CU); where even 64 x 64 tiles take two, the small
        // ones spread better.  Measured at 65 .. 511 rows on the layers of the small, base and large models: 1 024 -> 3 072 at 197
        // rows 5.9 us with 64 x 64 against 7.1 with 32 x 64 (336 of them) and 6.0 with 32 x 32 (672), at 394 rows (336 / 624 /
        // 1 248) 10.3 / 10.1 / 8.5; 4 096 -> 1 024 at 394 rows 9.9 with 32 x 64 against 11.8 with 32 x 32 (416).
        const int64_t rt = (g.M + 31) / 32, t11 = rt * (g.N / 32), t12 = rt * ((g.N + 63) / 64);
        const int64_t t22 = static_cast<int64_t>((g.M + 63) / 64) * ((g.N + 63) / 64);
        if constexpr (NQ == 0) {
            if (t11 <= cus || (t12 > cus && t22 > cus)) return launch_split<TOUT, 1, 1, 0>(g, w_hat, stream);
        }
        // (with the consumer's stage 1: 768 -> 3 072 at 197 rows 8.9 us with 64 x 64 against 10.7, at 394 rows 16.4 / 14.4)
        if (t12 <= cus || (t22 > cus && t12 <= 3 * cus)) return launch_split<TOUT, 1, 2, NQ>(g, w_hat, stream);
        return launch_split<TOUT, 2, 2, NQ>(g, w_hat, stream);
    }
    // 64 x 64 tiles (two workgroups on a CU) while they fit the chip at once, 128 x 128 beyond: measured crossovers between
    // 480 and 600 tiles at K = 384, 768 and 1 024 (384 -> 1 536 at 1 576 rows, 600 tiles: 7.9 against 6.9 us; 1 024 -> 3 072 at
    // 591 rows, 480 tiles: 9.2 against 11.5).  64 x 128 was never the fastest (one workgroup per CU for its LDS).
    const int64_t t64 = static_cast<int64_t>((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (t64 <= 2 * cus) return launch_tile<64, 64, 2, 2, TOUT, NQ, F8>(g, w_hat, stream);
    return launch_tile<128, 128, 2, 4, TOUT, NQ, F8>(g, w_hat, stream);
}

}  // namespace

void launch_gemm_tile(const GemmArgs &g, const void *w_hat, hipStream_t stream)
{
    auto run = [&](auto f8c) {
        constexpr bool F8 = decltype(f8c)::value;
        if (g.next_thr) {
            if (g.bits == 4) pick<__half, 4, F8>(g, w_hat, stream);
            else if (g.bits == 3) pick<__half, 3, F8>(g, w_hat, stream);
            else pick<__half, 2, F8>(g, w_hat, stream);
        } else if (g.y_f16) {
            pick<__half, 0, F8>(g, w_hat, stream);
        } else {
            pick<float, 0, F8>(g, w_hat, stream);
        }
    };
    if (g.fp8) run(std::true_type{});
    else run(std::false_type{});
}

}  // namespace arcq

using namespace arcq;

// Column blocks and the tile kernels up to the size where a workgroup of the weight-stationary kernels has five row blocks
// (one workgroup per compute unit).  Measured at M = 591 .. 25 216 on all layers of the tiny, small, base and large models,
// fp16 and FP8: the tile kernels win or tie at every shape with four or fewer (3 152 x 768 x 3 072: 31 against 35 us) and
// lose at every one with five or more (1 576 x 3 072 x 768 with fc2's stage 1: 30 against 25; 6 304 x 768 x 3 072: 55 / 43).
ARCQ_API int arcq_prepared_row_major(int64_t M, int64_t N, int64_t K)
{
    (void)K;
    if (N % 32 != 0) return 1;
    if (M < 512) return 0;
    const int64_t slabs = (N + 127) / 128, blocks = (M + 31) / 32;
    const int64_t ranges = std::min<int64_t>(std::max<int64_t>(device_cus() / slabs, 1), blocks);
    return (blocks + ranges - 1) / ranges >= 5 ? 1 : 0;
}

ARCQ_API int arcq_prepared_quant_row_major(int64_t M, int64_t N, int64_t K, int fp8)
{
    return gemm_quant_pays(M, N, K, fp8 != 0) ? 0 : arcq_prepared_row_major(M, N, K);
}

ARCQ_API int arcq_linear_prepared(const arcq_linear_prepared_args *a, void *stream)
{
    if (!a) return fail(ARCQ_ERR_NULL, "arcq_linear_prepared: args must not be NULL");
    if (a->M < 0 || a->N < 0 || a->K <= 0) return fail(ARCQ_ERR_SHAPE, "arcq_linear_prepared: bad sizes");
    if (a->K % 64 != 0 || (!a->w_row_major && a->N % 32 != 0))
        return fail(ARCQ_ERR_SHAPE, "arcq_linear_prepared: needs K a multiple of 64 and N a multiple of 32 (column blocks) (got N=%lld K=%lld)",
                    static_cast<long long>(a->N), static_cast<long long>(a->K));
    if (a->y_dtype != ARCQ_F16 && a->y_dtype != ARCQ_F32) return fail(ARCQ_ERR_DTYPE, "arcq_linear_prepared: y must be float16 or float32");
    if ((a->next_thresholds == nullptr) != (a->next_codebook == nullptr))
        return fail(ARCQ_ERR_NULL, "arcq_linear_prepared: next_thresholds and next_codebook go together");
    if (a->next_thresholds && (a->y_dtype != ARCQ_F16 || a->N % 64 != 0 || a->residual || !bits_ok(a->next_bits)))
        return fail(ARCQ_ERR_UNSUPPORTED, "arcq_linear_prepared: quantizing the output for the next layer needs float16, N a multiple of 64, "
                    "2/3/4 bits and no residual");
    if (a->M * a->N == 0) return ARCQ_OK;
    if (!a->x_hat || !a->w_hat || !a->y) return fail(ARCQ_ERR_NULL, "arcq_linear_prepared: NULL tensor pointer");
    if (a->M >= (int64_t(1) << 26) || a->N >= (int64_t(1) << 26) || a->M * a->K >= (int64_t(1) << 31) || a->N * a->K >= (int64_t(1) << 31))
        return fail(ARCQ_ERR_SHAPE, "arcq_linear_prepared: tensor too large");
    if (!aligned(a->x_hat, 16) || !aligned(a->w_hat, 16) || !aligned(a->y, 16) || !aligned(a->residual, 16))
        return fail(ARCQ_ERR_ALIGN, "arcq_linear_prepared: x_hat, w_hat, y and residual must be 16-byte aligned");
    GemmArgs g{a->x_hat, nullptr, nullptr, nullptr, nullptr, nullptr, a->bias, a->y, a->y_dtype == ARCQ_F16, static_cast<int>(a->M),
               static_cast<int>(a->N), static_cast<int>(a->K), a->next_thresholds ? a->next_bits : 4};
    g.residual = a->residual;
    g.gelu = a->activation == ARCQ_ACT_GELU;
    g.next_thr = a->next_thresholds;
    g.next_cb = a->next_codebook;
    g.fp8 = a->fp8 != 0;
    if (g.fp8) {
        if (!(a->w_mult > 0.0f)) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_linear_prepared: w_mult must be positive");
        g.fp8_inv = 1.0f / a->w_mult;
    }
    if (g.next_thr && !a->w_row_major && gemm_quant_pays(a->M, a->N, a->K, g.fp8)) {
        launch_gemm_quant(g, a->w_hat, static_cast<hipStream_t>(stream));
        return launch_status("arcq_linear_prepared");
    }
    if (g.fp8) {
        if (a->w_row_major) launch_gemm_fp8(g, a->w_hat, static_cast<hipStream_t>(stream));
        else launch_gemm_tile(g, a->w_hat, static_cast<hipStream_t>(stream));
        return launch_status("arcq_linear_prepared");
    }
    if (a->w_row_major) {
        if (a->M < 512) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_linear_prepared: row-major weights need 512 rows or more");
        launch_gemm_slab8(g, a->w_hat, static_cast<hipStream_t>(stream));
    } else {
        launch_gemm_tile(g, a->w_hat, static_cast<hipStream_t>(stream));
    }
    return launch_status("arcq_linear_prepared");
}
