// The MLP half of a transformer block in ONE launch, for many rows: a workgroup owns 64 rows of x and keeps everything between
// the block's skip connection and its output on its compute unit,
//
//   y = x + fc2( stage1( GELU( fc1( stage1( LayerNorm( x ) ) ) ) ) )          x, y [M, K] fp16, hidden width H = 4 K
//
// PROJ: the attention's output layer first, x = (the block's input) + proj( stage1( attention's output ) ).  A launch of its own of 64-row
// tiles is mostly what surrounds its short product (launch, tables, weight share, wait), all of which the one below pays anyway; its
// rows go to the LayerNorm through the LDS tile that held its x_hat, and to y, from where the last epilogue reads them back.
// 12 608 rows: K = 384 15.4 + 64.0 -> 76.2 us, K = 768 29.3 + 159 -> 181 (small model at 64 images 1 440 -> 1 381 us, base model
// 3 363 -> 3 340).
//
// Why beside the one-launch layer kernels (arcq_otf_rows.hip), which do the same as two launches: those write GELU's output (M x H
// values) and read it back, pay launch, table and weight-share set-up twice, and have little to overlap: a layer's product waits for
// its quantizer.  Here the hidden row is made 256 columns at a time and consumed at once, and the eight waves are two sets of four (a
// wave of each set on every SIMD) that take turns: while one set turns its 256 columns into x_hat (bias, GELU, the quantizer: vector
// ALU), the other multiplies (fc2 of the chunk before, fc1 of the chunk behind).  Measured on this chip a matrix instruction takes
// about two issue slots of the vector ALU's, so the two overlap nearly fully where waves are in different phases.
//
// A wave's fc1 tile is 64 rows x 64 columns, i.e. one quantization group of every row, 2 x 2 MFMA blocks.  The lanes l and l + 32 hold
// a row's columns in turns of four; one v_permlane32_swap per register gives lane l the whole group of row l, and the quantizer runs
// on a lane per group without a trip through LDS.
//
// The arithmetic, the order of every sum and the roundings are those of the two layers run one after the other: y has their bits.
//
// Measured: 12 608 rows, K = 768, fc1 and fc2 as two launches 110 + 120 us, this one 160 (the base model's forward at 64 images 3 809 ->
// 3 364 us); K = 384 29 + 39 -> 68 (1 559 -> 1 470); K = 192 -> 34 (a block 79 -> 69).  Clocks of a workgroup with proj in front, K =
// 768: 358 000 in all: set-up 20 000 (inputs from memory, shares of weights), proj's stage 1 and the wait 16 000, proj with its epilogue
// 31 700, LayerNorm and stage 1 29 500 (vector ALU, on two waves a SIMD), the first chunk of fc1 21 000, twelve steps of 16 800 to
// 20 200 (18 500 on average), the last product and output 17 500.  In a step the quantizing wave takes 3 700 for the rest of GELU,
// 7 500 to 8 900 for the quantizer and 4 400 to 5 100 for fc2's 96 MFMAs (3 072 at full rate), its partner 3 450 for those, 7 700 for
// fc1's 192 (6 144) and 3 000 for the first three eighths of GELU: a wave alone issues a vector instruction every five clocks or so, and
// the other's MFMAs take about eight of them each.  K = 384: 156 000, of them six steps of 12 600 to 14 800.
// Registers: all 256.  K = 768 keeps 19 to 22 more in scratch, a dozen of its loads and stores a step; K = 384 with proj two.
//
// Weights: rebuilt by the launch's workgroups between them, as in arcq_otf_rows.hip (proj's and fc1's together); fc2's under
// the first fc1 chunk, by the set that has nothing to multiply yet.
#include "arcq_act_quant_core.h"
#include "arcq_common.h"
#include "arcq_gemm.h"
#include "arcq_rows_share.h"

#include <type_traits>

namespace arcq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

struct MlpParams {
    const __half *x;                              // [M,K]
    const __half *attn;                           // [M,K], proj's input (PROJ)
    const float *thr0, *cb0;                      // activation thresholds / codebooks of proj (PROJ),
    const float *thr1, *cb1, *thr2, *cb2;         // fc1 and fc2
    float eps;
    const float *gamma, *beta;                    // LayerNorm weight / bias (fp32)
    float ln_eps;
    WeightShare w0, w1, w2;
    unsigned long long *counter;                  // two words: proj's and fc1's shares, fc2's
    long long wait_ticks;                         // as in arcq_otf_rows.hip
    unsigned long long *timeouts;
    const float *bias0, *bias1, *bias2;           // [K], [H], [K], or nullptr
    __half *y;
    int M;
};

constexpr int kWaves = 8, kSet = 4;               // waves of a workgroup, of a set
constexpr int kChunk = 64 * kSet;                 // hidden columns at a time
constexpr int kHiddenPitch = kChunk * 2 + 16;     // bytes per row of the hidden chunk in LDS
constexpr int kOutRow = 80;                       // bytes per staged output row: 32 fp16 + 16

constexpr int mlp_row_pitch(int G) { return 64 * G * 2 + 16; }
constexpr int mlp_lds_bytes(int G) { return 64 * mlp_row_pitch(G) + 64 * kHiddenPitch + 5 * 64 * G * 4; }      // beside the tables
constexpr int kBias0At = 24 * 1024;
static_assert(64 * 25 * 4 <= 64 * kHiddenPitch, "the LayerNorm's partial sums lie where the hidden chunk will be");
static_assert(kWaves * 32 * kOutRow <= kBias0At && kBias0At + 768 * 4 <= 64 * kHiddenPitch, "so do the output staging and, behind it, proj's bias");

// acc += x_hat[64 rows][GROUPS groups] * w_hat[NB blocks of 32 columns]^T.  `xs`: this lane's first piece of the x_hat tile in LDS (rows
// `PITCH` bytes apart); `w`: the first block (uniform), the blocks `stride` bytes apart, `at`: this lane's piece of it.  The fragments
// of DEPTH k-steps are in flight, the first DEPTH requested by start(), those of x_hat are read AHEAD k-steps early: few waves
// multiply at a time.
template <int NB, int GROUPS, int PITCH, int DEPTH, int AHEAD>
struct TileProduct {
    static constexpr int kSteps = 4 * GROUPS;
    u32x4_t ring[DEPTH][NB];
    __device__ __forceinline__ void fetch(u32x4_t (&r)[NB], const char *w, uint32_t at, int64_t stride, int s)
    {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            // An address in scalar registers, made here; else they are all made ahead, in vector registers.  (The barrier hides where
            // the pointer comes from, so its type says that it is global memory.)
            const auto *base = reinterpret_cast<const __attribute__((address_space(1))) char *>(reinterpret_cast<uintptr_t>(w) + nb * stride + (s >> 2) * 4096);
            asm("" : "+s"(base));
            r[nb] = *reinterpret_cast<const __attribute__((address_space(1))) u32x4_t *>(base + (s & 3) * 512 + at);
        }
    }
    __device__ __forceinline__ void start(const char *w, uint32_t at, int64_t stride)
    {
        asm volatile("" : "+v"(at));      // (a 32-bit offset beside the scalar address)
#pragma unroll
        for (int s = 0; s < DEPTH; ++s) fetch(ring[s], w, at, stride, s);
    }
    __device__ __forceinline__ void forget()      // (what start() requested is not used: no registers from here to the next start())
    {
#pragma unroll
        for (int s = 0; s < DEPTH; ++s)
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) asm volatile("" : "=v"(ring[s][nb]));
    }
    template <int USED>      // blocks, at most NB
    __device__ __forceinline__ void run(const unsigned char *xs, const char *w, uint32_t at, int64_t stride, float16_t (&acc)[NB][2])
    {
        asm volatile("" : "+v"(at));
        half8_t xf[AHEAD + 1][2];
        auto rows = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
                xf[s % (AHEAD + 1)][rb] = *reinterpret_cast<const half8_t *>(xs + (s >> 2) * 128 + (s & 3) * 16 + rb * 32 * PITCH);
        };
#pragma unroll
        for (int s = 0; s < AHEAD; ++s) rows(s);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            if (s + AHEAD < kSteps) rows(s + AHEAD);
#pragma unroll
            for (int nb = 0; nb < USED; ++nb) {
                half8_t wf;
                __builtin_memcpy(&wf, &ring[s % DEPTH][nb], 16);
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
                    acc[nb][rb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf, xf[s % (AHEAD + 1)][rb], acc[nb][rb], 0, 0, 0);
            }
            if (s + DEPTH < kSteps) fetch(ring[s % DEPTH], w, at, stride, s + DEPTH);
#pragma unroll
            for (int q = 0; q < 2 * USED; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                        // 1 MFMA
                if (q < 2 && s + AHEAD < kSteps) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);       // 1 LDS read
                if ((q & 1) && s + DEPTH < kSteps) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);     // 1 global load
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
};

// Waits (a bounded time) until the counter shows that all workgroups have written their shares; one thread.
__device__ __forceinline__ bool shares_written(const MlpParams &p, const unsigned long long *counter, unsigned long long target)
{
    bool ok = p.wait_ticks > 0;      // (a bound of zero: give up without looking -- how the tests reach the rebuild)
    const long long t0 = wall_clock64();
    while (ok && __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
        if (wall_clock64() - t0 > p.wait_ticks) {
            ok = false;
            break;
        }
        __builtin_amdgcn_s_sleep(4);
    }
    if (!ok) __hip_atomic_fetch_add(p.timeouts, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return ok;
}
__device__ __forceinline__ unsigned long long count_share(unsigned long long *counter)      // returns the value at which all are there
{
    const unsigned long long inc = blockIdx.x == 0 ? kEpoch - (gridDim.x - 1) : 1ull;
    const unsigned long long old = __hip_atomic_fetch_add(counter, inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return (old & ~(kEpoch - 1)) + kEpoch;
}
// Pieces lo, lo + step, ... < hi, AT_ONCE of them in flight.
template <int BITS, int G, int AT_ONCE>
__device__ __forceinline__ void rebuild_pieces(const WeightShare &w, int64_t lo, int64_t hi, int step)
{
    for (int64_t i0 = lo; i0 < hi; i0 += static_cast<int64_t>(AT_ONCE) * step) {
        Piece pc[AT_ONCE];
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j)
            if (i0 + static_cast<int64_t>(j) * step < hi) fetch_piece<BITS, G>(w, i0 + static_cast<int64_t>(j) * step, pc[j]);
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j)
            if (i0 + static_cast<int64_t>(j) * step < hi) finish_piece<BITS>(w, i0 + static_cast<int64_t>(j) * step, pc[j]);
    }
}

// G = K / 64.  PROJ: x is proj's output plus the skip connection, made here first.
template <int BITS, int G, bool PROJ>
__global__ void __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(2, 2)))
otf_mlp_kernel(const MlpParams p)
{
    constexpr int K = 64 * G, H = 4 * K, HG = 4 * G, CHUNKS = H / kChunk;
    constexpr int TILES = 2 * G, ROUNDS = (TILES + kWaves - 1) / kWaves;      // stage-1 tiles of 32 rows x one group, per wave
    constexpr int BLOCKS = K / 32, NB = (BLOCKS + kWaves - 1) / kWaves;       // fc2's column blocks, per wave (block wave + 8 nb)
    constexpr int PITCH = mlp_row_pitch(G);
    constexpr int kDepth1 = NB == 3 ? 4 : 6, kDepth2 = kDepth1, kAhead = 2;         // k-steps of weights in flight, of x_hat
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int s_ok;

    // (declared, not cut out of the dynamic LDS, whose address the compiler learns after it has chosen its instructions: a lookup's
    // constant part is then in the instruction and not an addition, 797 vector instructions for a row of 64 values where it took 925;
    // small model at 64 images 1 457 -> 1 434 us, base model the same)
    __shared__ QuantTables s_tables[PROJ ? 3 : 2];
    QuantTables &q1 = s_tables[0], &q2 = s_tables[1], &q0 = s_tables[PROJ ? 2 : 0];
    unsigned char *xs = smem;                                              // x_hat of proj, then x, then x_hat of fc1: [64][PITCH]
    unsigned char *hs = xs + 64 * PITCH;                                   // x_hat of fc2, one chunk: [64][kHiddenPitch]
    float *s_bias1 = reinterpret_cast<float *>(hs + 64 * kHiddenPitch);    // [H]
    float *s_bias2 = s_bias1 + H;                                          // [K]
    float *s_bias0 = reinterpret_cast<float *>(hs + kBias0At);             // [K] (PROJ)
    float *part = reinterpret_cast<float *>(hs);                           // the LayerNorm's partial sums: [64][2 G + 1]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), set = wave / kSet;
    const int lr = lane & 31, lh = lane >> 5;
    const int64_t row_base = static_cast<int64_t>(blockIdx.x) * 64;

    // ---- set-up: the tables' parameters and this wave's stage-1 tiles are requested first; waves 1 and 2 (PROJ: and 3) build the
    // tables, the workgroup's share of fc1's (and proj's) weights is rebuilt by the others ----
    QuantParams params{};
    if (wave == 1) params = load_quant_params<BITS>(p.thr1, p.cb1, lane);
    if (wave == 2) params = load_quant_params<BITS>(p.thr2, p.cb2, lane);
    if (PROJ && wave == 3) params = load_quant_params<BITS>(p.thr0, p.cb0, lane);
    const int row = lane >> 1, half = lane & 1;
    uint4 raws[ROUNDS][4];
#pragma unroll
    for (int rnd = 0; rnd < ROUNDS; ++rnd) {
        const int t = min(wave + rnd * kWaves, TILES - 1), rb = t / G, g = t - rb * G;
        const int64_t r0 = min(row_base + rb * 32 + row, static_cast<int64_t>(p.M) - 1);       // (rows past the end: the last one again)
        const __half *src = (PROJ ? p.attn : p.x) + r0 * K + g * 64 + half * 32;
#pragma unroll
        for (int i = 0; i < 4; ++i) raws[rnd][i] = *reinterpret_cast<const uint4 *>(src + i * 8);
    }
    constexpr int64_t kPieces = static_cast<int64_t>(H) * (K / 8);         // of either layer
    int64_t per = (kPieces + gridDim.x - 1) / gridDim.x;
    per = (per + 7) & ~int64_t(7);                                         // whole 128-byte lines per workgroup
    const int64_t share_lo = blockIdx.x * per, share_hi = min(share_lo + per, kPieces);
    constexpr int64_t kPieces0 = static_cast<int64_t>(K) * (K / 8);        // of proj
    const int64_t per0 = ((kPieces0 + gridDim.x - 1) / gridDim.x + 7) & ~int64_t(7);
    const int64_t share0_lo = blockIdx.x * per0, share0_hi = min(share0_lo + per0, kPieces0);
    constexpr int kAllBiases = H + (PROJ ? 2 : 1) * K;
    constexpr int kBiases = (kAllBiases + 64 * kWaves - 1) / (64 * kWaves);     // (all in flight at once: one after the other they take 5 us)
    float bias[kBiases];
#pragma unroll
    for (int i = 0; i < kBiases; ++i) {
        const int n = tid + i * 64 * kWaves;
        const float *b = n < H ? p.bias1 : n < H + K ? p.bias2 : p.bias0;
        bias[i] = b && n < kAllBiases ? b[n < H ? n : n < H + K ? n - H : n - H - K] : 0.0f;
    }
    if (wave == 1) build_quant_tables<BITS>(params, q1, lane);
    else if (wave == 2) build_quant_tables<BITS>(params, q2, lane);
    else if (PROJ && wave == 3) build_quant_tables<BITS>(params, q0, lane);
    else {
        constexpr int kBuilders = PROJ ? 3 : 2;
        const int64_t at = (wave == 0 ? 0 : wave - kBuilders) * 64 + lane;
        if constexpr (PROJ) rebuild_pieces<BITS, G, 2>(p.w0, share0_lo + at, share0_hi, 64 * (kWaves - kBuilders));
        rebuild_pieces<BITS, G, 4>(p.w1, share_lo + at, share_hi, 64 * (kWaves - kBuilders));
    }
#pragma unroll
    for (int i = 0; i < kBiases; ++i) {
        const int n = tid + i * 64 * kWaves;
        if (n < H + K) s_bias1[n] = bias[i];
        else if (n < kAllBiases) s_bias0[n - H - K] = bias[i];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                       // the written-through pieces have reached memory
    __syncthreads();
    unsigned long long target = 0;
    if (tid == 0) target = count_share(p.counter);

    auto tile_of = [&](int rnd, int &rb, int &g) {
        const int t = wave + rnd * kWaves;
        rb = t / G, g = t - rb * G;
        return t < TILES;
    };
    auto widened = [&](const uint4 (&raw)[4], float (&v)[32]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t w4[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
            widen(w4, v + 8 * i, 4);
        }
    };
    auto stage1 = [&](float (&v)[32], const QuantTables &q, unsigned char *dst) __attribute__((always_inline)) {
        float mu, var, s, sum;
        group_stats32x2(v, p.eps, mu, var, s);
        group_codes32x2<BITS>(v, mu, var, s, q, q.geometry, q.usable != 0, sum);
        const float code_mean = sum * 0.015625f;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            u32x4_t o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 8 * q4 + 2 * e;
                const __half2 h = __floats2half2_rn(fma_f32(s, v[j] - code_mean, mu), fma_f32(s, v[j + 1] - code_mean, mu));
                o[e] = *reinterpret_cast<const uint32_t *>(&h);
            }
            *reinterpret_cast<u32x4_t *>(dst + q4 * 16) = o;
        }
    };
    // (one wave drops whatever the caches may hold of the workspaces, before anyone reads them)
    auto await_shares = [&]() __attribute__((always_inline)) {
        if (tid == 0) s_ok = shares_written(p, p.counter, target);
        if (wave == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        __syncthreads();                          // x_hat is complete in LDS; s_ok is set
        if (!s_ok) {                              // workgroup-uniform
            if constexpr (PROJ) rebuild_pieces<BITS, G, 1>(p.w0, tid, kPieces0, 64 * kWaves);
            rebuild_pieces<BITS, G, 1>(p.w1, tid, kPieces, 64 * kWaves);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
    };
    const unsigned char *x_lane = xs + lr * PITCH + lh * 64;
    const uint32_t at = lh * 2048 + lr * 16;
    const int blocks = (BLOCKS - wave + kWaves - 1) / kWaves;                // of proj's and fc2's columns: wave, wave + 8, ...
    // The rows of x (or of y) that the epilogues below add, in the order in which a wave writes its blocks.
    auto skip_rows = [&](const __half *x, u32x4_t (&skip)[NB][2][2]) __attribute__((always_inline)) {
        int l = lane;
        asm volatile("" : "+v"(l));      // (the addresses are made twice; else they are kept in registers from the first use to the last)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t grow = min(row_base + i * 16 + (l >> 2), static_cast<int64_t>(p.M) - 1);
                const int c0 = min(wave + nb * kWaves, BLOCKS - 1) * 32;
                skip[nb][i >> 1][i & 1] = *reinterpret_cast<const u32x4_t *>(x + grow * K + c0 + (l & 3) * 8);
            }
    };
    // Bias, rounding, skip connection; a wave's 32 x 32 block at a time through its staging tile.  put(row of the tile, column, 8 values).
    auto epilogue = [&](const float16_t (&acc)[NB][2], const float *bias, const u32x4_t (&skip)[NB][2][2], auto put) __attribute__((always_inline)) {
        unsigned char *stage = hs + wave * 32 * kOutRow;
        int l = lane;
        asm volatile("" : "+v"(l));
        const int lr = l & 31, lh = l >> 5;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (nb >= blocks) break;
            const int c0 = (wave + nb * kWaves) * 32;
#pragma unroll
            for (int rb = 0; rb < 2; ++rb) {
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const float4 b = *reinterpret_cast<const float4 *>(bias + c0 + 8 * t + 4 * lh);
                    u32x2_t pk;
                    pk[0] = half_pair(acc[nb][rb][4 * t] + b.x, acc[nb][rb][4 * t + 1] + b.y);
                    pk[1] = half_pair(acc[nb][rb][4 * t + 2] + b.z, acc[nb][rb][4 * t + 3] + b.w);
                    *reinterpret_cast<u32x2_t *>(stage + lr * kOutRow + (8 * t + 4 * lh) * 2) = pk;
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int r = i * 16 + (l >> 2);
                    const u32x4_t v = *reinterpret_cast<const u32x4_t *>(stage + r * kOutRow + (l & 3) * 16);
                    float a[8], b[8];
                    u32x4_t o;
                    widen(reinterpret_cast<const uint32_t *>(&v), a, 4);
                    widen(reinterpret_cast<const uint32_t *>(&skip[nb][rb][i]), b, 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[e] = half_pair(a[2 * e] + b[2 * e], a[2 * e + 1] + b[2 * e + 1]);
                    put(rb * 32 + r, c0 + (l & 3) * 8, o);
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
    };

    // ---- PROJ: stage 1 of attention's output, proj, the skip connection: the block's x in y and, row by row, in xs ----
    if constexpr (PROJ) {
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) {
            int rb, g;
            if (!tile_of(rnd, rb, g)) break;
            float v[32];
            widened(raws[rnd], v);
            stage1(v, q0, xs + (rb * 32 + row) * PITCH + g * 128 + half * 64);
        }
        await_shares();
        float16_t acc0[NB][2];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc0[nb][rb][v] = 0.0f;
        const char *w0 = reinterpret_cast<const char *>(p.w0.out) + static_cast<int64_t>(BLOCKS < kWaves ? min(wave, BLOCKS - 1) : wave) * (K * 64);
        const int64_t last0 = BLOCKS % kWaves == 0 || blocks == NB ? static_cast<int64_t>(kWaves) * K * 64 : 0;
        TileProduct<NB, G, PITCH, kDepth2, kAhead> proj;
        proj.start(w0, at, last0);
        if (BLOCKS % kWaves == 0 || blocks == NB) proj.template run<NB>(x_lane, w0, at, last0, acc0);
        else proj.template run<NB - 1>(x_lane, w0, at, last0, acc0);
        __builtin_amdgcn_sched_barrier(0);
        u32x4_t skip[NB][2][2];
        skip_rows(p.x, skip);
        __syncthreads();                          // everyone is done with proj's x_hat
        epilogue(acc0, s_bias0, skip, [&](int r, int c, const u32x4_t &o) __attribute__((always_inline)) {
            *reinterpret_cast<u32x4_t *>(xs + r * PITCH + c * 2) = o;
            if (row_base + r < p.M) *reinterpret_cast<u32x4_t *>(p.y + (row_base + r) * K + c) = o;      // (read again at the end, by this lane)
        });
        __syncthreads();
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) {
            int rb, g;
            if (!tile_of(rnd, rb, g)) break;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                raws[rnd][i] = *reinterpret_cast<const uint4 *>(xs + (rb * 32 + row) * PITCH + g * 128 + half * 64 + i * 16);
        }
    }

    // ---- LayerNorm (arithmetic and summation order of otf_rows_kernel) and stage 1 into xs ----
    {
        float xv[ROUNDS][32];
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) widened(raws[rnd], xv[rnd]);
        constexpr float fk = static_cast<float>(K);
        constexpr int ppitch = 2 * G + 1;
        float stat[ROUNDS];
        auto row_totals = [&]() {                // stat: this lane's partial sums in, its rows' sums out
#pragma unroll
            for (int rnd = 0; rnd < ROUNDS; ++rnd) {
                int rb, g;
                if (tile_of(rnd, rb, g)) part[(rb * 32 + row) * ppitch + 2 * g + half] = stat[rnd];
            }
            __syncthreads();
#pragma unroll
            for (int rnd = 0; rnd < ROUNDS; ++rnd) {
                int rb, g;
                float acc = 0.0f;
                if (tile_of(rnd, rb, g))
                    for (int i = 0; i < 2 * G; ++i) acc += part[(rb * 32 + row) * ppitch + i];
                stat[rnd] = acc;
            }
            __syncthreads();
        };
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) {
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) a += xv[rnd][j];
            stat[rnd] = a;
        }
        row_totals();
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) {
            const float mean = stat[rnd] / fk;
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                xv[rnd][j] -= mean;
                const float sq = xv[rnd][j] * xv[rnd][j];
                s += sq;
            }
            stat[rnd] = s;
        }
        row_totals();
#pragma unroll
        for (int rnd = 0; rnd < ROUNDS; ++rnd) {
            int rb, g;
            if (!tile_of(rnd, rb, g)) break;
            const float rstd = 1.0f / sqrtf(stat[rnd] / fk + p.ln_eps);
            const float4 *gp = reinterpret_cast<const float4 *>(p.gamma + g * 64 + half * 32);
            const float4 *bp = reinterpret_cast<const float4 *>(p.beta + g * 64 + half * 32);
            float (&v)[32] = xv[rnd];
#pragma unroll
            for (int j4 = 0; j4 < 8; ++j4) {
                const float4 gv = gp[j4], bv = bp[j4];
                const float g4[4] = {gv.x, gv.y, gv.z, gv.w}, b4[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float t = v[4 * j4 + e] * rstd;
                    const float u = t * g4[e];
                    v[4 * j4 + e] = __half2float(__float2half_rn(u + b4[e]));
                }
            }
            stage1(v, q1, xs + (rb * 32 + row) * PITCH + g * 128 + half * 64);
        }
    }
    if constexpr (PROJ) __syncthreads();
    else await_shares();

    // ---- the chunks.  Step t: one set quantizes chunk t of the hidden row, then adds chunk t - 1 to fc2's sums; the other one adds
    // chunk t - 1, multiplies chunk t + 1 of fc1 and takes the first kEarly eighths of its GELU, so that both are done at about the
    // same time and the matrix units and vector ALUs of every SIMD have work side by side.  Then they change places. ----
    // (Base model at 64 images 3 369 us; half of GELU instead 3 389, five eighths 3 442.  Small model 1 394; all of it 1 400.)
    constexpr int kEarly = G >= 12 ? 3 : 5;
    constexpr int64_t stride1 = static_cast<int64_t>(K) * 64, stride2 = static_cast<int64_t>(kWaves) * H * 64;
    const unsigned char *h_lane = hs + lr * kHiddenPitch + lh * 64;
    const char *w1 = reinterpret_cast<const char *>(p.w1.out) + (wave % kSet) * 2 * stride1;
    // (K = 192: six blocks.  The last two waves use none, but request one with the others.)
    const char *w2 = reinterpret_cast<const char *>(p.w2.out) + static_cast<int64_t>(BLOCKS < kWaves ? min(wave, BLOCKS - 1) : wave) * (H * 64);
    float16_t acc[NB][2];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int rb = 0; rb < 2; ++rb)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[nb][rb][v] = 0.0f;
    TileProduct<NB, kChunk / 64, kHiddenPitch, kDepth2, kAhead> fc2;
    uint32_t pairs[32];
    const int64_t last2 = BLOCKS % kWaves == 0 || blocks == NB ? stride2 : 0;      // (a wave with fewer blocks reads one of them again)
    auto add_chunk = [&](int c) __attribute__((always_inline)) {
        if (BLOCKS % kWaves == 0 || blocks == NB) fc2.template run<NB>(h_lane, w2 + c * (kChunk / 64 * 4096), at, last2, acc);
        else fc2.template run<NB - 1>(h_lane, w2 + c * (kChunk / 64 * 4096), at, last2, acc);
    };
    for (int t = -1;; ++t) {
        const bool mine = t >= 0 && t < CHUNKS && set == (t & 1);
        if (mine) {
            gelu_pairs<kEarly, 8>(pairs);
            quantize_row<BITS, false>(pairs, q2, p.eps, pairs);
            fc2.start(t >= 1 ? w2 + (t - 1) * (kChunk / 64 * 4096) : w1, at, last2);      // (at t = 0 nothing: unused, but never what is not yet written)
        }
        if (t >= 1) add_chunk(t - 1);
        if (t == CHUNKS) break;
        if (!mine && t + 1 < CHUNKS && set == ((t + 1) & 1)) {
            float16_t tile[2][2];
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
#pragma unroll
                for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                    for (int v = 0; v < 16; ++v) tile[cb][rb][v] = 0.0f;
            TileProduct<2, G, PITCH, kDepth1, kAhead> fc1;
            const char *w = w1 + static_cast<int64_t>(t + 1) * (kChunk / 32) * stride1;
            fc1.start(w, at, stride1);
            fc1.template run<2>(x_lane, w, at, stride1, tile);
            tile_to_rows<false>(tile, 1.0f, s_bias1 + (t + 1) * kChunk + (wave % kSet) * 64, lane, pairs);
            gelu_pairs<0, kEarly>(pairs);
        } else if (t == -1) {
            rebuild_pieces<BITS, HG, 3>(p.w2, share_lo + (wave % kSet) * 64 + lane, share_hi, 64 * kSet);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if (t == 0) {
            if (tid == 64 * kSet) s_ok = shares_written(p, p.counter + 1, target);
            if (wave == kSet) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        __syncthreads();                         // chunk t - 1 has been consumed
        if (t == -1) {
            if (tid == 64 * kSet) target = count_share(p.counter + 1);
            fc2.forget();
            continue;
        }
        if (mine) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                u32x4_t o;
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = pairs[4 * i + e];
                *reinterpret_cast<u32x4_t *>(hs + lane * kHiddenPitch + (wave % kSet) * 128 + i * 16) = o;
            }
        }
        if (t == 0 && !s_ok) {
            rebuild_pieces<BITS, HG, 1>(p.w2, tid, kPieces, 64 * kWaves);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        if (mine || t == CHUNKS - 1) fc2.start(w2 + t * (kChunk / 64 * 4096), at, last2);
        else fc2.forget();
        __syncthreads();                         // chunk t is complete
    }
    u32x4_t skip[NB][2][2];
    skip_rows(PROJ ? p.y : p.x, skip);
    __syncthreads();                             // (the staging tiles lie where the last chunk was)
    epilogue(acc, s_bias2, skip, [&](int r, int c, const u32x4_t &o) __attribute__((always_inline)) {
        if (row_base + r < p.M) store_streaming16(p.y + (row_base + r) * K + c, o[0], o[1], o[2], o[3]);
    });
}

template <int BITS, int G, bool PROJ>
int launch_mlp(const MlpParams &p, hipStream_t stream)
{
    constexpr int lds = mlp_lds_bytes(G);
    static_assert(lds + (PROJ ? 3 : 2) * sizeof(QuantTables) <= 160 * 1024 - 64, "does not fit");
    allow_dynamic_lds<otf_mlp_kernel<BITS, G, PROJ>>(lds);
    const int tiles = (p.M + 63) / 64;
    if (resident_workgroups<otf_mlp_kernel<BITS, G, PROJ>>(64 * kWaves, lds) < tiles) return kNotLaunched;
    hipLaunchKernelGGL((otf_mlp_kernel<BITS, G, PROJ>), dim3(tiles), dim3(64 * kWaves), lds, stream, p);
    return launch_status("arcq_mlp_otf");
}
template <int BITS, bool PROJ>
int launch_mlp_k(const MlpParams &p, int64_t K, hipStream_t stream)
{
    switch (K) {
    case 192: return launch_mlp<BITS, 3, PROJ>(p, stream);
    case 256: return launch_mlp<BITS, 4, PROJ>(p, stream);
    case 384: return launch_mlp<BITS, 6, PROJ>(p, stream);
    default: return launch_mlp<BITS, 12, PROJ>(p, stream);
    }
}
template <int BITS>
int launch_mlp_proj(const MlpParams &p, int64_t K, hipStream_t stream)
{
    return p.attn ? launch_mlp_k<BITS, true>(p, K, stream) : launch_mlp_k<BITS, false>(p, K, stream);
}

}  // namespace
}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_mlp_otf_supported(int64_t M, int64_t K, int64_t H)
{
    if (K != 192 && K != 256 && K != 384 && K != 768) return 0;
    return M >= 512 && H == 4 * K && (M + 63) / 64 <= device_cus() ? 1 : 0;
}

ARCQ_API int arcq_mlp_otf_pays(int64_t M, int64_t K, int64_t H)
{
    if (!arcq_mlp_otf_supported(M, K, H) || tuning().gemm_kernel) return 0;
    if (const char *e = tuning().rows) return e[0] != '0';
    // (the launch takes as long however few its workgroups are; figures beside the block's launches, arcq_host.cpp)
    return M > (K == 192 ? 6600 : K == 256 ? 7200 : K == 384 ? 8700 : 10240);
}

ARCQ_API int arcq_mlp_otf(const arcq_mlp_args *a, void *stream)
{
    if (!a) return fail(ARCQ_ERR_NULL, "arcq_mlp_otf: NULL arguments");
    if (!bits_ok(a->bits)) return fail(ARCQ_ERR_BITS, "arcq_mlp_otf: bits must be 2, 3, or 4");
    if (a->M < 0 || a->K < 0 || a->H < 0) return fail(ARCQ_ERR_SHAPE, "arcq_mlp_otf: negative size");
    if (!arcq_mlp_otf_supported(a->M, a->K, a->H)) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_mlp_otf: sizes not served");
    const arcq_mlp_layer *const l[3] = {&a->fc1, &a->fc2, &a->proj};
    const int layers = a->attn ? 3 : 2;
    if (!a->x || !a->y || !a->ln_weight || !a->ln_bias) return fail(ARCQ_ERR_NULL, "arcq_mlp_otf: NULL tensor pointer");
    for (int i = 0; i < layers; ++i) {
        const arcq_mlp_layer *f = l[i];
        if (!f->a_thresholds || !f->a_codebook || !f->packed_w || !f->w_codebook || !f->w_center || !f->w_scale || !f->w_code_sum || !f->w_hat_ws)
            return fail(ARCQ_ERR_NULL, "arcq_mlp_otf: NULL tensor pointer");
        if (!aligned(f->packed_w, 4) || !aligned(f->w_hat_ws, 128))
            return fail(ARCQ_ERR_ALIGN, "arcq_mlp_otf: packed_w must be 4-byte, w_hat_ws 128-byte aligned");
    }
    if (a->y == a->x || a->y == a->attn) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_mlp_otf: y must not alias x or attn");
    if (!aligned(a->attn, 16) || !aligned(a->x, 16) || !aligned(a->y, 16) || !aligned(a->ln_weight, 16) || !aligned(a->ln_bias, 16))
        return fail(ARCQ_ERR_ALIGN, "arcq_mlp_otf: x, attn, y, ln_weight and ln_bias must be 16-byte aligned");
    MlpParams p{};
    p.x = static_cast<const __half *>(a->x), p.y = static_cast<__half *>(a->y);
    p.attn = static_cast<const __half *>(a->attn);
    p.thr0 = a->proj.a_thresholds, p.cb0 = a->proj.a_codebook;
    p.thr1 = a->fc1.a_thresholds, p.cb1 = a->fc1.a_codebook, p.thr2 = a->fc2.a_thresholds, p.cb2 = a->fc2.a_codebook;
    p.eps = a->eps, p.gamma = a->ln_weight, p.beta = a->ln_bias, p.ln_eps = a->ln_eps;
    WeightShare *w[3] = {&p.w1, &p.w2, &p.w0};
    for (int i = 0; i < layers; ++i)
        *w[i] = WeightShare{l[i]->packed_w, l[i]->w_codebook, l[i]->w_center, l[i]->w_scale, l[i]->w_code_sum, static_cast<__half *>(l[i]->w_hat_ws)};
    p.bias0 = a->proj.bias, p.bias1 = a->fc1.bias, p.bias2 = a->fc2.bias;
    p.M = static_cast<int>(a->M);
    p.counter = rows_counters_for(a->fc1.w_hat_ws, &p.timeouts);
    if (!p.counter) return fail(ARCQ_ERR_UNSUPPORTED, "arcq_mlp_otf: no counter left for this workspace");
    p.wait_ticks = tuning().rows_wait_ticks;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int rc = a->bits == 4 ? launch_mlp_proj<4>(p, a->K, st) : a->bits == 3 ? launch_mlp_proj<3>(p, a->K, st) : launch_mlp_proj<2>(p, a->K, st);
    return rc == kNotLaunched ? fail(ARCQ_ERR_UNSUPPORTED, "arcq_mlp_otf: the device does not hold all workgroups at once") : rc;
}
