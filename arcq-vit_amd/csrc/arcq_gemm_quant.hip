// Stages 2+3 on prepared operands with the next layer's stage 1 at the end, for many rows: x_hat' = stage1'( [GELU] ( x_hat * w_hat^T +
// bias ) ), x_hat and x_hat' in the 32-row block layout, w_hat in the 32-column block layout; fp16 or FP8 operands.
//
// Why beside gemm_pair_kernel / gemm_fp8_kernel, which end the same way: there a workgroup's waves share slices of K through barriers, so
// all of them multiply and then all of them quantize, and the epilogue (some 40 vector instructions a value: GELU and the quantizer)
// adds to the products.  Here a workgroup keeps 64 columns of w_hat, all of K, in LDS for good (128 KB at K = 1 024): after the first
// copy there is no barrier, every wave walks 64-row tiles of its own and the waves of a SIMD drift apart, so that one's epilogue runs
// under the others' products.  64 columns are one group of the next layer: see tile_to_rows.
//
// x_hat streams from L2 into registers, each 1 KB fragment for two MFMAs: 64 bytes a clock and compute unit at the full matrix rate, a
// little more than L1 gives (60); with the epilogue the launch needs half of that.  The weights cost LDS 64 of its 128 bytes a clock.
// The order of the k-steps per output is that of the other kernels: the same bits.
//
// Measured: 50 432 x 1 024 -> 4 096 with GELU 580 -> 478 us (414 without the epilogue: 35 % of the vector ALU's time hides), 25 216 x
// 768 -> 3 072 198 -> 159, FP8 6 304 x 768 -> 3 072 47.9 -> 35.2.  Two units of x_hat in flight instead of one: 526 -> 494; without the
// stores 460; three waves a SIMD spill: 612.
#include "arcq_act_quant_core.h"
#include "arcq_common.h"
#include "arcq_gemm.h"

#include <algorithm>

namespace arcq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWaves = 8;                   // two a SIMD, of 256 registers (three of 168 spill: 528 -> 612 us)
constexpr int kAhead = 2;                   // units of x_hat in flight
constexpr int kSlabAt = 64 * 4;             // (the bias first)
constexpr int kUnitBytes = 4096;            // 32 rows (columns) x 128 bytes of an operand
constexpr int quant_lds_bytes(int units) { return kSlabAt + 2 * units * kUnitBytes; }      // beside the tables
constexpr int kMaxLds = 160 * 1024 - static_cast<int>(sizeof(QuantTables)) - 16;

struct QuantArgs {
    const char *x;              // 32-row block layout, rows of 128 `units` bytes
    const char *w;              // 32-column block layout
    const float *bias;          // [N] or nullptr
    char *y;                    // 32-row block layout of the next operand, rows of out_bytes
    const float *thr, *cb;
    float inv_mult, eps;
    int M, N, units, gelu;
    int streaming;              // the output will not be found in a cache again
    int slabs, ranges, tiles_per_range;      // 64 columns; row ranges; 64-row tiles
};

template <int BITS, bool F8>
__global__ void __launch_bounds__(64 * kWaves)
gemm_quant_kernel(const QuantArgs a)
{
    constexpr int kSteps = F8 ? 2 : 4;       // MFMA k-steps of a unit
    constexpr int kLoads = 4 / kSteps;       // 16-byte pieces a lane reads for one
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    // (declared, not cut out of the dynamic LDS, whose address the compiler learns after it has chosen its instructions: a lookup's
    // constant part is then in the instruction and not an addition: large model at 256 images 41.2 -> 41.0 ms)
    __shared__ QuantTables tables;
    float *s_bias = reinterpret_cast<float *>(smem);
    unsigned char *slab = smem + kSlabAt;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 31, lh = lane >> 5;

    // Each XCD (workgroups are dealt to the eight round-robin) takes a run of (row range, slab), slabs fastest: its workgroups walk the
    // same rows at about the same time and read them through one L2.
    const int jobs = a.slabs * a.ranges, per_xcd = (jobs + 7) / 8;
    const int job = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || job >= jobs) return;
    const int range = job / a.slabs, n0 = (job - range * a.slabs) * 64;
    const int tile_rows = (a.M + 63) / 64;
    const int first = range * a.tiles_per_range, last = min(first + a.tiles_per_range, tile_rows);

    // ---- the slab, tables and bias into LDS ----
    const int slab_bytes = 2 * a.units * kUnitBytes;
    {
        QuantParams params{};
        if (wave == 0) params = load_quant_params<BITS>(a.thr, a.cb, lane);
        const char *src = a.w + static_cast<int64_t>(n0 / 32) * a.units * kUnitBytes;
        for (int p = wave * 1024; p < slab_bytes; p += kWaves * 1024)      // (whole kilobytes)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + p + lane * 16),
                                             (__attribute__((address_space(3))) void *)(slab + p), 16, 0, 0);
        if (tid < 64) s_bias[tid] = a.bias ? a.bias[n0 + tid] : 0.0f;
        if (wave == 0) build_quant_tables<BITS>(params, tables, lane);
        __builtin_amdgcn_s_waitcnt(0x0F70);      // vmcnt(0)
        asm volatile("" ::: "memory");
        __syncthreads();
    }

    // A tile's two row blocks: base of the first unit, distance of its pieces (16 bytes a row; the last block's rows lie compactly) and
    // this lane's offset.  Fragments: unit u, step s, piece e of this lane is piece 8 u + F(s, e) of its row, F = 4 lh + s (fp16) or
    // 4 s + 2 lh + e (FP8).
    const int blocks = (a.M + 31) / 32;
    struct Rows {
        const char *base[2];
        int step[2];
        uint32_t at[2];
    };
    auto rows_of = [&](int tile) __attribute__((always_inline)) {
        Rows r;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            const int blk = min(2 * tile + rb, blocks - 1), rows = min(32, a.M - blk * 32);
            r.base[rb] = a.x + static_cast<int64_t>(blk) * a.units * kUnitBytes;
            r.step[rb] = rows * 16;
            r.at[rb] = static_cast<uint32_t>((F8 ? 2 : 4) * lh * r.step[rb] + min(lr, rows - 1) * 16);
        }
        return r;
    };
    u32x4_t xs[kAhead][4][2];
    auto fetch = [&](const Rows &r, int u, int slot, int i) __attribute__((always_inline)) {      // i = s * kLoads + e
        const int f = F8 ? 4 * (i >> 1) + (i & 1) : i;
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
            // (an address in scalar registers plus a 32-bit offset; the barrier hides where the pointer comes from, so its type says it)
            const auto *p = reinterpret_cast<const __attribute__((address_space(1))) char *>(
                reinterpret_cast<uintptr_t>(r.base[rb]) + static_cast<uint32_t>((8 * u + f) * r.step[rb]));
            asm("" : "+s"(p));
            uint32_t at = r.at[rb];
            asm("" : "+v"(at));
            xs[slot][i][rb] = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t *>(p + at);
        }
    };
    const unsigned char *w_lane = slab + lr * 16 + lh * (F8 ? 1024 : 2048);
    const int block_bytes = a.units * kUnitBytes;
    u32x4_t wf[2][2][kLoads];                // [step parity][column block][piece]
    auto weights = [&](int u, int s, int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int e = 0; e < kLoads; ++e)
                wf[slot][cb][e] = *reinterpret_cast<const u32x4_t *>(w_lane + cb * block_bytes + u * kUnitBytes + (F8 ? s * 2048 + e * 512 : s * 512));
    };

    const int out_bytes = F8 ? (a.N + 127) / 128 * 128 : a.N * 2;
    int tile = first + wave;
    if (tile >= last) return;
    Rows cur = rows_of(tile);
#pragma unroll
    for (int j = 0; j < kAhead; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) fetch(cur, j, j, i);
    weights(0, 0, 0);
    for (; tile < last; tile += kWaves) {
        const Rows next = rows_of(min(tile + kWaves, last - 1));
        mfma_block_t acc[2][2];
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[cb][rb][v] = 0.0f;
        for (int u0 = 0; u0 < a.units; u0 += kAhead) {
            const bool wrap = u0 + kAhead == a.units;      // (the next tile's first units)
            Rows from;
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
                from.base[rb] = wrap ? next.base[rb] : cur.base[rb], from.step[rb] = wrap ? next.step[rb] : cur.step[rb],
                from.at[rb] = wrap ? next.at[rb] : cur.at[rb];
            const int nu = wrap ? 0 : u0 + kAhead;
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
#pragma unroll
                for (int s = 0; s < kSteps; ++s) {
                    if (s + 1 < kSteps) weights(u0 + j, s + 1, (s + 1) & 1);
                    else weights(j + 1 < kAhead ? u0 + j + 1 : nu, 0, 0);
#pragma unroll
                    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                        for (int rb = 0; rb < 2; ++rb) {
                            if constexpr (F8) {
                                i32x8_t wv, xv;
                                __builtin_memcpy(&wv, &wf[s & 1][cb][0], 32);
                                __builtin_memcpy(&xv, &xs[j][2 * s][rb], 16);
                                __builtin_memcpy(reinterpret_cast<char *>(&xv) + 16, &xs[j][2 * s + 1][rb], 16);
                                acc[cb][rb] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wv, xv, acc[cb][rb], 0, 0, 0, 0, 0, 0);
                            } else {
                                half8_t wv, xv;
                                __builtin_memcpy(&wv, &wf[s & 1][cb][0], 16);
                                __builtin_memcpy(&xv, &xs[j][s][rb], 16);
                                acc[cb][rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wv, xv, acc[cb][rb], 0, 0, 0);
                            }
                        }
#pragma unroll
                    for (int e = 0; e < kLoads; ++e) fetch(from, nu + j, j, s * kLoads + e);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                       // 1 MFMA
                        if (q < 2) __builtin_amdgcn_sched_group_barrier(0x100, kLoads, 0);                       // LDS reads
                    }
                    __builtin_amdgcn_sched_group_barrier(0x020, 2 * kLoads, 0);                                  // global loads
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        // ---- epilogue: a row per lane ----
        uint32_t row[32], out[F8 ? 16 : 32];
        tile_to_rows<F8>(acc, a.inv_mult, s_bias, lane, row);
        if (a.gelu) gelu_pairs<0, 8>(row);
        quantize_row<BITS, F8>(row, tables, a.eps, out);
        const int blk = 2 * tile + lh, rows = min(32, a.M - blk * 32);
        if (blk < blocks && lr < rows) {
            char *dst = a.y + static_cast<int64_t>(blk) * 32 * out_bytes + (static_cast<int64_t>(F8 ? n0 / 16 : n0 / 8) * rows + lr) * 16;
#pragma unroll
            for (int i = 0; i < (F8 ? 4 : 8); ++i) {
                char *d = dst + static_cast<int64_t>(i) * rows * 16;
                if (a.streaming) store_streaming16(d, out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]);
                else store_writethrough16(d, out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]);
            }
            if (F8 && n0 + 64 == a.N && (a.N & 64) != 0) {      // (a row's padding to 128 values)
#pragma unroll
                for (int i = 4; i < 8; ++i) store_writethrough16(dst + static_cast<int64_t>(i) * rows * 16, 0, 0, 0, 0);
            }
        }
        cur = next;
    }
}

template <int BITS, bool F8>
void launch_quant(const QuantArgs &a, hipStream_t stream)
{
    allow_dynamic_lds<gemm_quant_kernel<BITS, F8>>(kMaxLds);
    const int jobs = a.slabs * a.ranges;
    hipLaunchKernelGGL((gemm_quant_kernel<BITS, F8>), dim3((jobs + 7) / 8 * 8), dim3(64 * kWaves), quant_lds_bytes(a.units), stream, a);
}

}  // namespace

namespace {
// Row ranges of 64-row tiles, one workgroup each for every 64 columns: as many as the compute units hold at once.
struct Ranges {
    int64_t count, tiles;      // tiles per range
};
Ranges ranges_of(int64_t tiles, int64_t slabs)
{
    const int64_t count = std::min(std::max(device_cus() / slabs, int64_t(1)), tiles);
    return {count, (tiles + count - 1) / count};
}
}  // namespace

// Measured beside the kernels that end the same way, in blocks (us a block at these rows; one after the other from a graph, with everything
// in the caches, the quotients are up to 5 % lower):
//   - At least 4.5 tiles of 64 x 64 a compute unit (1 576 rows: 1 024 -> 4 096 116 -> 109, 768 -> 3 072 86 -> 80, FP8 93 -> 88 and
//     75 -> 72; 985 rows, four tiles: 83 -> 86 and 69 -> 72).
//   - Six units of fp16 (K = 384) are too little work a tile to hide the epilogue under: 3 152 .. 9 456 rows 65.6 -> 64.0 .. 107 -> 106,
//     25 216 rows 207 -> 209; below 4.5 tiles it never pays.
//   - A range's ninth to twelfth tile is a third turn for its SIMDs, four tiles a turn.  The other kernels' workgroups (128 columns, more
//     often all of the chip) have eight blocks of 32 rows there or nine: eight are fewer.  5 122 rows: 384 -> 1 536 83.3 -> 80.6,
//     512 -> 1 536 108 -> 104, 768 -> 1 536 FP8 127 -> 121; 2 167 rows: 768 -> 3 328 114 -> 112, FP8 93.8 -> 92.0; three ranges, 1 576
//     rows: 768 -> 4 160 FP8 87.4 -> 85.5, fp16 102.8 / 102.8, 512 -> 4 160 83.3 / 87.2.  With fewer ranges the weights' way into LDS
//     counts for more, and this kernel's are half (1 182 rows: 768 -> 5 504 101.5 / 102, -> 10 240 at 788 rows 123 / 130).
//   - 129 slabs and a few more leave half of the chip idle (the others: 195 workgroups).  Long ranges: 768 -> 8 256 at 5 910 rows
//     380 -> 367, FP8 at 4 531 219 -> 210; short ones 123 / 128 at 1 182 rows; 160 slabs 230 / 250 at 2 758, FP8 1 024 -> 10 240
//     198 / 210 at 3 152; 257 slabs are two rounds in both.
bool gemm_quant_pays(int64_t M, int64_t N, int64_t K, bool fp8)
{
    const int units = operand_units(static_cast<int>(K), fp8);
    if (N % 64 != 0 || M < 512 || units < 6 || units % kAhead != 0 || quant_lds_bytes(units) > kMaxLds) return false;
    const int64_t rows = (M + 63) / 64, slabs = N / 64, tiles = rows * slabs, cus = device_cus();
    if (2 * tiles < 9 * cus || (!fp8 && units < 8 && tiles > 16 * cus)) return false;
    const Ranges r = ranges_of(rows, slabs);
    if (r.tiles > 64 && slabs <= cus && 16 * slabs * r.count < 9 * cus) return false;
    if (r.count >= (fp8 ? 3 : 4) && r.tiles > 8 && r.tiles <= 12) {
        const int64_t blocks = (M + 31) / 32, others = std::max(cus / ((N + 127) / 128), int64_t(1));
        if ((blocks + others - 1) / others <= 8) return false;
    }
    return true;
}

void launch_gemm_quant(const GemmArgs &g, const void *w_hat, hipStream_t stream)
{
    QuantArgs a{};
    a.x = static_cast<const char *>(g.x_hat), a.w = static_cast<const char *>(w_hat);
    a.bias = g.bias, a.y = static_cast<char *>(g.y);
    a.thr = g.next_thr, a.cb = g.next_cb;
    a.inv_mult = g.fp8_inv, a.eps = 1.0e-6f;
    a.M = g.M, a.N = g.N, a.units = operand_units(g.K, g.fp8), a.gelu = g.gelu ? 1 : 0;
    // Outputs of more than 200 MB (the memory-side cache has 256) leave with streaming stores: a block of 50 432 rows of 1 024 values
    // 1 653 -> 1 636 us, of 768 (310 MB) 1 070 -> 1 057; 25 216 rows of 768 (155 MB) 551 -> 557.
    a.streaming = static_cast<int64_t>(g.M) * g.N * (g.fp8 ? 1 : 2) > int64_t(200) << 20;
    a.slabs = g.N / 64;
    const Ranges r = ranges_of((g.M + 63) / 64, a.slabs);
    a.ranges = static_cast<int>(r.count), a.tiles_per_range = static_cast<int>(r.tiles);
    if (g.fp8) {
        if (g.bits == 4) launch_quant<4, true>(a, stream);
        else if (g.bits == 3) launch_quant<3, true>(a, stream);
        else launch_quant<2, true>(a, stream);
    } else {
        if (g.bits == 4) launch_quant<4, false>(a, stream);
        else if (g.bits == 3) launch_quant<3, false>(a, stream);
        else launch_quant<2, false>(a, stream);
    }
}

}  // namespace arcq
