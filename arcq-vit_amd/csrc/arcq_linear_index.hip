// Index-space linears: y = sum over groups of
//   gs*mu_x*mu_w + s_x*s_w*(sum_j P[xcode_j][wcode_j] - Sx*Sw/gs)
// with P = cb_a (x) cb_w, i.e. no reconstruction of either operand
// (EXT/arcq_linear_kernel.cu:22-78 for packed codes / fp64, :136-202 for byte
// codes / fp32).  These are the reference's "packed" and "u8" runtime formats.
// All kernels keep the reference's summation order per output, so that the result equals a
// serial CPU evaluation bit for bit; contraction is switched off for that reason.  Group size 64
// runs the tiled kernels further down; the two kernels right below take any group size.
#include "arcq_common.h"
#include "arcq_gemm.h"

#include <type_traits>

namespace arcq {

constexpr int kIdxTile = 16;  // 16 x 16 outputs per 256-thread workgroup (the any-group-size kernels)

// fp64 accumulation, codes extracted from the packed rows on the fly.
__global__ void __launch_bounds__(256)
linear_index_packed_kernel(const uint8_t *__restrict__ px, const float *__restrict__ xc, const float *__restrict__ xs,
                           const float *__restrict__ xcs, const uint8_t *__restrict__ pw,
                           const float *__restrict__ wc, const float *__restrict__ ws, const float *__restrict__ wcs,
                           const float *__restrict__ table, const float *__restrict__ bias, float *__restrict__ y,
                           int64_t rows, int64_t out_f, int64_t in_f, int bits, int gs, int levels)
{
#pragma clang fp contract(off)
    extern __shared__ float s_table[];
    for (int i = threadIdx.x; i < levels * levels; i += blockDim.x) s_table[i] = table[i];
    __syncthreads();
    const int64_t r = static_cast<int64_t>(blockIdx.y) * kIdxTile + (threadIdx.x >> 4);
    const int64_t o = static_cast<int64_t>(blockIdx.x) * kIdxTile + (threadIdx.x & 15);
    if (r >= rows || o >= out_f) return;
    const int64_t groups = in_f / gs;
    const int64_t pcols = packed_cols(in_f, bits);
    const uint8_t *__restrict__ xr = px + r * pcols;
    const uint8_t *__restrict__ wr = pw + o * pcols;
    double acc = bias ? static_cast<double>(bias[o]) : 0.0;
    for (int64_t g = 0; g < groups; ++g) {
        double cross = 0.0;
        const int64_t base = g * gs;
        for (int j = 0; j < gs; ++j) {
            const int a = get_code(xr, base + j, bits);
            const int b = get_code(wr, base + j, bits);
            cross += static_cast<double>(s_table[a * levels + b]);
        }
        const int64_t xm = r * groups + g, wm = o * groups + g;
        const double mu_term = static_cast<double>(gs) * static_cast<double>(xc[xm]) * static_cast<double>(wc[wm]);
        const double residual_term = static_cast<double>(xs[xm]) * static_cast<double>(ws[wm]) *
            (cross - (static_cast<double>(xcs[xm]) * static_cast<double>(wcs[wm])) / static_cast<double>(gs));
        acc += mu_term + residual_term;
    }
    y[r * out_f + o] = static_cast<float>(acc);
}

// fp32, byte codes.  The reference gives each output a 32-lane warp: lane l sums
// the table entries of j = l, l+32, ... and the 32 partials are folded by a
// shuffle-down tree (16, 8, 4, 2, 1).  Here one thread owns the output and
// evaluates the same 32 partials and the same tree in registers.
__global__ void __launch_bounds__(256)
linear_index_u8_kernel(const uint8_t *__restrict__ xcodes, const float *__restrict__ xc, const float *__restrict__ xs,
                       const float *__restrict__ xcs, const uint8_t *__restrict__ wcodes,
                       const float *__restrict__ wc, const float *__restrict__ ws, const float *__restrict__ wcs,
                       const float *__restrict__ table, const float *__restrict__ bias, float *__restrict__ y,
                       int64_t rows, int64_t out_f, int64_t in_f, int gs, int levels)
{
#pragma clang fp contract(off)
    extern __shared__ float s_table[];
    for (int i = threadIdx.x; i < levels * levels; i += blockDim.x) s_table[i] = table[i];
    __syncthreads();
    const int64_t r = static_cast<int64_t>(blockIdx.y) * kIdxTile + (threadIdx.x >> 4);
    const int64_t o = static_cast<int64_t>(blockIdx.x) * kIdxTile + (threadIdx.x & 15);
    if (r >= rows || o >= out_f) return;
    const int64_t groups = in_f / gs;
    const uint8_t *__restrict__ xr = xcodes + r * in_f;
    const uint8_t *__restrict__ wr = wcodes + o * in_f;
    float acc = bias ? bias[o] : 0.0f;
    for (int64_t g = 0; g < groups; ++g) {
        const int64_t base = g * gs;
        float p[32];
#pragma unroll
        for (int l = 0; l < 32; ++l) {
            float cross = 0.0f;
            for (int j = l; j < gs; j += 32)
                cross += s_table[static_cast<int>(xr[base + j]) * levels + static_cast<int>(wr[base + j])];
            p[l] = cross;
        }
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
#pragma unroll
            for (int l = 0; l < off; ++l) p[l] = p[l] + p[l + off];
        }
        const float cross = p[0];
        const int64_t xm = r * groups + g, wm = o * groups + g;
        const float mu_term = static_cast<float>(gs) * xc[xm] * wc[wm];
        const float residual_term = xs[xm] * ws[wm] * (cross - (xcs[xm] * wcs[wm]) / static_cast<float>(gs));
        acc += mu_term + residual_term;
    }
    y[r * out_f + o] = acc;
}

// ---- group size 64: tiled kernels -------------------------------------------------------------------------------
// A workgroup owns 16 rows x 64 outputs; a thread one row and four consecutive outputs.  Per group the tile's codes
// are fetched once (packed rows: `bits` bytes = eight codes per load, consecutive threads reading consecutive bytes),
// unpacked once into LDS as bytes -- x as [row][j], w transposed as [j][output], so that a thread's four weight codes
// of one j are a single dword read -- and every product-table lookup is one LDS read.  What fixes the result's bits is
// the order in which one output's terms are added; that is the reference's, per output: serial over j in fp64 for
// the packed format; for the byte format the 32 strided partial sums folded by the shuffle-down tree, which is
// evaluated here depth first (the same additions, associated the same way) so that only five values per output are live.
constexpr int kTileRows = 16, kTileOuts = 64;

// BITS = 2 / 3 / 4: packed codes, fp64 accumulation.  BITS = 0: byte codes, fp32, tree order.
// OPT = outputs per thread: four (256 threads per workgroup) for launches that fill the chip; one (1024 threads) for
// small ones, whose duration is the length of one thread's chain of additions (197 x 768 x 192: 156 tiles).
template <int BITS, int OPT>
__global__ void __launch_bounds__(1024 / OPT)
linear_index_tile_kernel(const uint8_t *__restrict__ xq, const float *__restrict__ xc, const float *__restrict__ xs,
                         const float *__restrict__ xcs, const uint8_t *__restrict__ wq,
                         const float *__restrict__ wc, const float *__restrict__ ws, const float *__restrict__ wcs,
                         const float *__restrict__ table, const float *__restrict__ bias, float *__restrict__ y,
                         int64_t rows, int64_t out_f, int64_t in_f, int levels)
{
#pragma clang fp contract(off)
    extern __shared__ float s_table[];
    __shared__ __attribute__((aligned(16))) uint8_t s_x[kTileRows][64];
    __shared__ __attribute__((aligned(16))) uint8_t s_w[64][kTileOuts];          // [j][output]
    constexpr int kOutsPerThread = OPT;
    constexpr int kThreads = 1024 / OPT;
    constexpr int kThreadsPerRow = kTileOuts / OPT;
    const int tid = threadIdx.x;
    for (int i = tid; i < levels * levels; i += kThreads) s_table[i] = table[i];
    const int tr = tid / kThreadsPerRow;                       // row of the tile
    const int to = (tid % kThreadsPerRow) * kOutsPerThread;    // first of this thread's outputs in the tile
    const int64_t r = static_cast<int64_t>(blockIdx.y) * kTileRows + tr;
    const int64_t o0 = static_cast<int64_t>(blockIdx.x) * kTileOuts + to;
    const int64_t groups = in_f / 64;
    const int64_t rc = r < rows ? r : rows - 1;    // rows / outputs past the end repeat the last one and are not stored
    constexpr int kRowBytes = BITS ? 8 * BITS : 64;      // bytes of one group in a row of codes
    const int64_t pcols = groups * kRowBytes;

    using acc_t = typename std::conditional<BITS != 0, double, float>::type;
    acc_t acc[kOutsPerThread];
    int64_t oc[kOutsPerThread];
#pragma unroll
    for (int i = 0; i < kOutsPerThread; ++i) {
        oc[i] = o0 + i < out_f ? o0 + i : out_f - 1;
        acc[i] = bias ? static_cast<acc_t>(bias[oc[i]]) : static_cast<acc_t>(0);
    }

    for (int64_t g = 0; g < groups; ++g) {
        __syncthreads();          // the previous group's codes have been used (first round: the table is complete)
        // ---- this group's codes into LDS, unpacked ----
        if constexpr (BITS != 0) {
            if (tid < kTileRows * 8) {                               // x: 16 rows x 8 chunks of eight codes
                const int row = tid >> 3, ch = tid & 7;
                const int64_t rr = static_cast<int64_t>(blockIdx.y) * kTileRows + row;
                const uint32_t w8 = load_codes8<BITS>(xq + (rr < rows ? rr : rows - 1) * pcols + g * kRowBytes + ch * BITS);
                uint32_t lo = 0, hi = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    lo |= ((w8 >> (BITS * q)) & ((1u << BITS) - 1u)) << (8 * q);
                    hi |= ((w8 >> (BITS * (q + 4))) & ((1u << BITS) - 1u)) << (8 * q);
                }
                *reinterpret_cast<uint2 *>(&s_x[row][ch * 8]) = make_uint2(lo, hi);
            }
            for (int job = tid; job < kTileOuts * 8; job += kThreads) {      // w: 64 outputs x 8 chunks of eight codes
                const int out = job >> 3, ch = job & 7;
                const int64_t oo = static_cast<int64_t>(blockIdx.x) * kTileOuts + out;
                const uint32_t w8 = load_codes8<BITS>(wq + (oo < out_f ? oo : out_f - 1) * pcols + g * kRowBytes + ch * BITS);
#pragma unroll
                for (int q = 0; q < 8; ++q) s_w[ch * 8 + q][out] = static_cast<uint8_t>((w8 >> (BITS * q)) & ((1u << BITS) - 1u));
            }
        } else {
            if (tid < 256) {                                         // x: 16 rows x 64 bytes, one dword per thread
                const int row = tid >> 4, c4 = (tid & 15) * 4;
                const int64_t rr = static_cast<int64_t>(blockIdx.y) * kTileRows + row;
                *reinterpret_cast<uint32_t *>(&s_x[row][c4]) =
                    *reinterpret_cast<const uint32_t *>(xq + (rr < rows ? rr : rows - 1) * pcols + g * 64 + c4);
            }
            if (tid < 256) {                                         // w: 64 outputs x 64 bytes, sixteen bytes per thread
                const int out = tid >> 2, c16 = (tid & 3) * 16;
                const int64_t oo = static_cast<int64_t>(blockIdx.x) * kTileOuts + out;
                const uint4 v = *reinterpret_cast<const uint4 *>(wq + (oo < out_f ? oo : out_f - 1) * pcols + g * 64 + c16);
                const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int q = 0; q < 16; ++q) s_w[c16 + q][out] = static_cast<uint8_t>(d[q >> 2] >> (8 * (q & 3)));
            }
        }
        __syncthreads();
        // one j for this thread's row and its four outputs: the table entries P[x code][w code]
        auto entries = [&](int j, float (&e)[kOutsPerThread]) __attribute__((always_inline)) {
            const int a = static_cast<int>(s_x[tr][j]) * levels;
            if constexpr (OPT == 4) {
                const uint32_t wb = *reinterpret_cast<const uint32_t *>(&s_w[j][to]);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) e[i] = s_table[a + static_cast<int>((wb >> (8 * i)) & 255u)];
            } else {
                e[0] = s_table[a + static_cast<int>(s_w[j][to])];
            }
        };
        acc_t cross[kOutsPerThread];
        if constexpr (BITS != 0) {
#pragma unroll
            for (int i = 0; i < kOutsPerThread; ++i) cross[i] = 0.0;
#pragma unroll 8
            for (int j = 0; j < 64; ++j) {
                float e[kOutsPerThread];
                entries(j, e);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) cross[i] += static_cast<double>(e[i]);
            }
        } else {
            // leaf l = the partial sum of lane l: j = l, then j = l + 32; node(level, l) = what lane l holds after the
            // fold with offset 32 >> level (lane l adds lane l + offset): node(5, 0) is the group's sum.
            auto leaf = [&](int l, float (&p)[kOutsPerThread]) __attribute__((always_inline)) {
                float e0[kOutsPerThread], e1[kOutsPerThread];
                entries(l, e0);
                entries(l + 32, e1);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) {
                    float c = 0.0f;
                    c += e0[i];
                    c += e1[i];
                    p[i] = c;
                }
            };
            auto node1 = [&](int l, float (&v)[kOutsPerThread]) __attribute__((always_inline)) {      // offset 16
                float b[kOutsPerThread];
                leaf(l, v);
                leaf(l + 16, b);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) v[i] = v[i] + b[i];
            };
            auto node2 = [&](int l, float (&v)[kOutsPerThread]) __attribute__((always_inline)) {      // offset 8
                float b[kOutsPerThread];
                node1(l, v);
                node1(l + 8, b);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) v[i] = v[i] + b[i];
            };
            auto node3 = [&](int l, float (&v)[kOutsPerThread]) __attribute__((always_inline)) {      // offset 4
                float b[kOutsPerThread];
                node2(l, v);
                node2(l + 4, b);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) v[i] = v[i] + b[i];
            };
            auto node4 = [&](int l, float (&v)[kOutsPerThread]) __attribute__((always_inline)) {      // offset 2
                float b[kOutsPerThread];
                node3(l, v);
                node3(l + 2, b);
#pragma unroll
                for (int i = 0; i < kOutsPerThread; ++i) v[i] = v[i] + b[i];
            };
            float b[kOutsPerThread];
            node4(0, cross);                                                                             // offset 1
            node4(1, b);
#pragma unroll
            for (int i = 0; i < kOutsPerThread; ++i) cross[i] = cross[i] + b[i];
        }
        // ---- the group's closed form (EXT/arcq_linear_kernel.cu:65-74 / :187-197) ----
        const int64_t xm = rc * groups + g;
        const float xcv = xc[xm], xsv = xs[xm], xcsv = xcs[xm];
#pragma unroll
        for (int i = 0; i < kOutsPerThread; ++i) {
            const int64_t wm = oc[i] * groups + g;
            if constexpr (BITS != 0) {
                const double mu_term = 64.0 * static_cast<double>(xcv) * static_cast<double>(wc[wm]);
                const double residual_term = static_cast<double>(xsv) * static_cast<double>(ws[wm]) *
                    (cross[i] - (static_cast<double>(xcsv) * static_cast<double>(wcs[wm])) / 64.0);
                acc[i] += mu_term + residual_term;
            } else {
                const float mu_term = 64.0f * xcv * wc[wm];
                const float residual_term = xsv * ws[wm] * (cross[i] - (xcsv * wcs[wm]) / 64.0f);
                acc[i] += mu_term + residual_term;
            }
        }
    }
    if (groups == 0) __syncthreads();
    if (r < rows) {
#pragma unroll
        for (int i = 0; i < kOutsPerThread; ++i)
            if (o0 + i < out_f) y[r * out_f + o0 + i] = static_cast<float>(acc[i]);
    }
}

// ---- group size 64, the codebooks at hand -------------------------------------------------------------------------------
// What bounds the tiled kernel above is its table gather: two operands' address arithmetic and a conflicting 4-byte LDS
// read per product (random entries of a 256-entry table).  The product table of a layer is P[a][b] = RN32(cb_a[a] * cb_w[b]),
// so with the two codebooks at hand an entry is one multiplication of two decoded values.  Every workgroup checks that on
// the table it was given (levels^2 comparisons); where it does not hold the same loops run with the gather.
//
// A wave owns a tile of 8 R rows x 8 C outputs, a lane R x C of them (rows ly + 8 i, outputs lx + 8 k), and decodes the two
// operands of a group into its own LDS region, half a group (32 j) at a time: [j / 4][row or output][4], so that one 16-byte
// read brings four j of a row: 3 bytes of LDS reads per product at R = 2, C = 4.  What bounds it now is the
// vector pipe: multiply, (fp64: convert,) add per product, 71 of the 111 us of 1576 x 384 -> 1536; the decoding is the rest.
//
// The sum over j of one group does not depend on the other groups, so the waves of a workgroup share ONE tile and take the
// groups g = wave, wave + S, ...; only the terms they yield are added in the order of the groups, by all threads together,
// once per round of S groups.  That makes small launches S times shorter and leaves every addition where the reference has
// it: serial over j in fp64 for the packed format, the 32-lane tree for the byte format (eight j of one residue class mod
// 8 at a time, the classes in the order 0 4 2 6 1 5 3 7, which is the tree depth first), terms in ascending g.
// Measured, whole calls, this kernel against the tiled one: 1576 x 384 -> 1536 (4 bits) 111 against 186 us, 12608 rows 744
// against 1172; 1576 x 768 -> 768 108 / 207; byte codes 394 x 768 -> 768 35 / 86, 12608 x 384 -> 1536 546 / 1177.
constexpr int kIdxMinWaves = 3, kIdxMaxWaves = 4;
constexpr int kIdxRegion = 32 * 33 * 8;            // bytes per wave: operands of half a group, then its terms (33-double pitch)

struct IndexArgs {
    const uint8_t *xq;
    const float *xc, *xs, *xcs;
    const uint8_t *wq;
    const float *wc, *ws, *wcs, *table, *a_cb, *w_cb, *bias;
    float *y;
    int rows, out_f, G, levels;
    // linear_index_mfma_kernel, where the table does not qualify: the workgroups that share the tiles, and how many behind them take
    // one of the last tiles each
    int workers, singles;
};

// The product table and the codebooks in LDS.
template <int LEVELS>
struct IndexTables {
    float table[LEVELS * LEVELS], a_cb[LEVELS], w_cb[LEVELS];
};
// Stores entry i; whether it is the product of its two codebook values.
template <int LEVELS>
__device__ __forceinline__ int index_table_entry(const IndexArgs &p, IndexTables<LEVELS> &t, int i, float value)
{
    t.table[i] = value;
    if (i < p.levels) t.a_cb[i] = p.a_cb[i], t.w_cb[i] = p.w_cb[i];
    return static_cast<int>(__float_as_uint(value) == __float_as_uint(p.a_cb[i / p.levels] * p.w_cb[i % p.levels]));
}

// The tile of rows r0 .. and outputs o0 .., by a workgroup of at least MINW waves.  FILL: the tables are loaded here; otherwise they
// are complete, and `outer` says whether the product table is one of the codebooks.
template <int BITS, int R, int C, int MINW, bool FILL>
__device__ __forceinline__ void index_wide_tile(const IndexArgs &p, int r0, int o0, IndexTables<BITS ? 1 << BITS : 16> &tables, int outer)
{
#pragma clang fp contract(off)
    constexpr bool kPacked = BITS != 0;
    constexpr int TR = 8 * R, TC = 8 * C;
    constexpr int kRowBytes = kPacked ? 8 * BITS : 64;
    constexpr int kPieceBytes = kRowBytes / 8;                        // eight codes
    constexpr int kPieceDwords = kPacked ? 1 : 2;
    constexpr int kXJobs = TR * 8 / 64, kWJobs = TC * 8 / 64;          // pieces per lane and group
    constexpr int kPitch = TC + 1;                                     // terms per row of the tile
    using acc_t = typename std::conditional<kPacked, double, float>::type;
    static_assert((TR + TC) * 32 * 4 <= kIdxRegion && TR * kPitch * static_cast<int>(sizeof(acc_t)) <= kIdxRegion, "LDS region");
    const float *s_table = tables.table, *s_acb = tables.a_cb, *s_wcb = tables.w_cb;
    extern __shared__ __attribute__((aligned(16))) unsigned char idx_smem[];     // [S waves][kIdxRegion]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nthreads = blockDim.x, S = nthreads >> 6;
    const int lx = lane & 7, ly = lane >> 3;
    const int rows = p.rows, out_f = p.out_f, G = p.G, levels = p.levels;
    const uint8_t *__restrict__ xq = p.xq, *__restrict__ wq = p.wq;
    const float *__restrict__ xc = p.xc, *__restrict__ xs = p.xs, *__restrict__ xcs = p.xcs, *__restrict__ wc = p.wc, *__restrict__ ws = p.ws;
    const float *__restrict__ wcs = p.wcs, *__restrict__ bias = p.bias;
    float *__restrict__ y = p.y;
    unsigned char *region = idx_smem + wave * kIdxRegion;
    float *s_x = reinterpret_cast<float *>(region), *s_w = s_x + TR * 32;

    // Pieces: job i of a lane is row lane % T, piece (lane / T) + i * (64 / T) of the group (T = TR or TC; rows past the end
    // repeat the last one and are not stored).
    const uint8_t *x_src = xq + static_cast<int64_t>(min(r0 + lane % TR, rows - 1)) * G * kRowBytes + (lane / TR) * kPieceBytes;
    const uint8_t *w_src = wq + static_cast<int64_t>(min(o0 + lane % TC, out_f - 1)) * G * kRowBytes + (lane / TC) * kPieceBytes;
    uint32_t xn[kXJobs][kPieceDwords], wn[kWJobs][kPieceDwords];
    auto load_piece = [](const uint8_t *p, uint32_t (&d)[kPieceDwords]) __attribute__((always_inline)) {
        if constexpr (kPacked) {
            d[0] = load_codes8<BITS>(p);
        } else {
            const uint2 v = *reinterpret_cast<const uint2 *>(p);
            d[0] = v.x;
            d[1] = v.y;
        }
    };
    auto fetch = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kXJobs; ++i) load_piece(x_src + static_cast<int64_t>(g) * kRowBytes + i * (64 / TR) * kPieceBytes, xn[i]);
#pragma unroll
        for (int i = 0; i < kWJobs; ++i) load_piece(w_src + static_cast<int64_t>(g) * kRowBytes + i * (64 / TC) * kPieceBytes, wn[i]);
    };
    if (wave < G) fetch(wave);
    if constexpr (FILL) {
        int same = 1;
        for (int i = tid; i < levels * levels; i += nthreads) same &= index_table_entry(p, tables, i, p.table[i]);
        outer = __syncthreads_and(same);
    }
    // With its address seen by an asm statement the region is memory the statements in the loops below may touch, so its
    // reads stay where they are written.  (The compiler otherwise moves all reads of a group to its top: 500 registers.)
    asm volatile("" ::"v"(region) : "memory");

    // The outputs this thread sums: TR * TC of them over the workgroup, consecutive in a row.
    constexpr int kSums = (TR * TC + 64 * MINW - 1) / (64 * MINW);
    acc_t acc[kSums];
#pragma unroll
    for (int i = 0; i < kSums; ++i) {
        const int p = i * nthreads + tid, o = o0 + p % TC;
        acc[i] = (bias && p < TR * TC && o < out_f) ? static_cast<acc_t>(bias[o]) : static_cast<acc_t>(0);
    }

    auto body = [&](auto outer_c) __attribute__((always_inline)) {
        constexpr bool OUTER = decltype(outer_c)::value;
        // An operand's decoded value: its codebook entry, or (gather) its share of the byte offset of the table entry.
        auto x_value = [&](uint32_t c) __attribute__((always_inline)) { return OUTER ? s_acb[c] : __uint_as_float(c * static_cast<uint32_t>(levels) * 4u); };
        auto w_value = [&](uint32_t c) __attribute__((always_inline)) { return OUTER ? s_wcb[c] : __uint_as_float(c * 4u); };
        auto product = [&](float xv, float wv) __attribute__((always_inline)) {
            if constexpr (OUTER) return xv * wv;
            else return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(s_table) + (__float_as_uint(xv) + __float_as_uint(wv)));
        };
        // Half `h` of a group into LDS.  Packed: j = 32 h ... + 31, slot jq = (j % 32) / 4.  Bytes: the classes j % 8 = h' + {0, 4,
        // 2, 6} with h' = h, class number n (0..3) and piece p at slot 2 n + p / 4.
        auto put = [&](float *dst, int T, auto jobs_c, const uint32_t (*codes)[kPieceDwords], int h, auto value) __attribute__((always_inline)) {
            constexpr int JOBS = decltype(jobs_c)::value;
            const int row = lane % T, p0 = lane / T;
#pragma unroll
            for (int i = 0; i < JOBS; ++i) {
                const int p = p0 + i * (64 / T);
                if constexpr (kPacked) {
                    if ((p >> 2) == h) {
                        float v[8];
#pragma unroll
                        for (int q = 0; q < 8; ++q) v[q] = value((codes[i][0] >> (BITS * q)) & ((1u << BITS) - 1u));
                        float *d = dst + ((p & 3) * 2 * T + row) * 4;
                        *reinterpret_cast<float4 *>(d) = make_float4(v[0], v[1], v[2], v[3]);
                        *reinterpret_cast<float4 *>(d + T * 4) = make_float4(v[4], v[5], v[6], v[7]);
                    }
                } else {
#pragma unroll
                    for (int n = 0; n < 4; ++n) {
                        const uint32_t d = (n & 1) ? codes[i][kPieceDwords - 1] : codes[i][0];      // bytes 4.. / 0..3
                        const uint32_t c = (d >> (8 * (h + (n & 2)))) & 255u;
                        dst[((2 * n + (p >> 2)) * T + row) * 4 + (p & 3)] = value(c);
                    }
                }
            }
        };
        const int rounds = (G + S - 1) / S;
        for (int round = 0; round < rounds; ++round) {
            const int g = round * S + wave;
            if (g < G) {
                uint32_t xk[kXJobs][kPieceDwords], wk[kWJobs][kPieceDwords];
#pragma unroll
                for (int i = 0; i < kXJobs; ++i)
#pragma unroll
                    for (int d = 0; d < kPieceDwords; ++d) xk[i][d] = xn[i][d];
#pragma unroll
                for (int i = 0; i < kWJobs; ++i)
#pragma unroll
                    for (int d = 0; d < kPieceDwords; ++d) wk[i][d] = wn[i][d];
                if (g + S < G) fetch(g + S);
                acc_t cross[R][C];
#pragma unroll
                for (int r = 0; r < R; ++r)
#pragma unroll
                    for (int c = 0; c < C; ++c) cross[r][c] = 0;
#pragma unroll 1
                for (int h = 0; h < 2; ++h) {
                    put(s_x, TR, std::integral_constant<int, kXJobs>{}, xk, h, x_value);
                    put(s_w, TC, std::integral_constant<int, kWJobs>{}, wk, h, w_value);
                    asm volatile("" ::: "memory");          // (wave-private LDS: operations execute in order)
                    if constexpr (kPacked) {
#pragma unroll 1
                        for (int jq = 0; jq < 8; ++jq) {
                            float4 xv[R], wv[C];
#pragma unroll
                            for (int r = 0; r < R; ++r) xv[r] = *reinterpret_cast<const float4 *>(s_x + (jq * TR + ly + 8 * r) * 4);
#pragma unroll
                            for (int c = 0; c < C; ++c) wv[c] = *reinterpret_cast<const float4 *>(s_w + (jq * TC + lx + 8 * c) * 4);
                            const float *xf = reinterpret_cast<const float *>(xv), *wf = reinterpret_cast<const float *>(wv);
#pragma unroll
                            for (int q = 0; q < 4; ++q)
#pragma unroll
                                for (int r = 0; r < R; ++r)
#pragma unroll
                                    for (int c = 0; c < C; ++c) cross[r][c] += static_cast<double>(product(xf[4 * r + q], wf[4 * c + q]));
                        }
                    } else {
                        float n3a[R][C];                     // the sum of this half's first two classes (offset 4)
#pragma unroll 1
                        for (int pair = 0; pair < 2; ++pair) {
                            float n2a[R][C];
#pragma unroll
                            for (int e = 0; e < 2; ++e) {
                                const int n = 2 * pair + e;
                                float4 xv[R][2];
#pragma unroll
                                for (int r = 0; r < R; ++r)
#pragma unroll
                                    for (int k = 0; k < 2; ++k) xv[r][k] = *reinterpret_cast<const float4 *>(s_x + ((2 * n + k) * TR + ly + 8 * r) * 4);
#pragma unroll
                                for (int c = 0; c < C; ++c) {
                                    float4 wv[2];
#pragma unroll
                                    for (int k = 0; k < 2; ++k) wv[k] = *reinterpret_cast<const float4 *>(s_w + ((2 * n + k) * TC + lx + 8 * c) * 4);
                                    const float w0[4] = {wv[0].x, wv[0].y, wv[0].z, wv[0].w}, w1[4] = {wv[1].x, wv[1].y, wv[1].z, wv[1].w};
#pragma unroll
                                    for (int r = 0; r < R; ++r) {
                                        const float x0[4] = {xv[r][0].x, xv[r][0].y, xv[r][0].z, xv[r][0].w}, x1[4] = {xv[r][1].x, xv[r][1].y, xv[r][1].z, xv[r][1].w};
                                        float leaf[4];       // lanes c, c + 8, c + 16, c + 24 of the class
#pragma unroll
                                        for (int q = 0; q < 4; ++q) leaf[q] = product(x0[q], w0[q]) + product(x1[q], w1[q]);
                                        const float n2 = (leaf[0] + leaf[2]) + (leaf[1] + leaf[3]);     // offsets 16, 8
                                        if (e == 0) n2a[r][c] = n2;
                                        else n2a[r][c] += n2;                                             // offset 4
                                    }
                                }
                                asm volatile("" ::: "memory");
                            }
#pragma unroll
                            for (int r = 0; r < R; ++r)
#pragma unroll
                                for (int c = 0; c < C; ++c) {
                                    if (pair == 0) {
                                        n3a[r][c] = n2a[r][c];
                                    } else {
                                        const float n4 = n3a[r][c] + n2a[r][c];                           // offset 2
                                        cross[r][c] = h == 0 ? n4 : cross[r][c] + n4;                     // offset 1
                                    }
                                }
                        }
                    }
                    asm volatile("" ::: "memory");
                }
                // ---- the group's closed form (EXT/arcq_linear_kernel.cu:65-74 / :187-197), into the wave's LDS region ----
                acc_t *term = reinterpret_cast<acc_t *>(region);
                float wcv[C], wsv[C], wmv[C];
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int64_t wm = static_cast<int64_t>(min(o0 + lx + 8 * c, out_f - 1)) * G + g;
                    wcv[c] = wc[wm], wsv[c] = ws[wm], wmv[c] = wcs[wm];
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int64_t xm = static_cast<int64_t>(min(r0 + ly + 8 * r, rows - 1)) * G + g;
                    const float xcv = xc[xm], xsv = xs[xm], xcsv = xcs[xm];
#pragma unroll
                    for (int c = 0; c < C; ++c) {
                        acc_t v;
                        if constexpr (kPacked) {
                            const double mu_term = 64.0 * static_cast<double>(xcv) * static_cast<double>(wcv[c]);
                            const double residual_term = static_cast<double>(xsv) * static_cast<double>(wsv[c]) *
                                (cross[r][c] - (static_cast<double>(xcsv) * static_cast<double>(wmv[c])) / 64.0);
                            v = mu_term + residual_term;
                        } else {
                            const float mu_term = 64.0f * xcv * wcv[c];
                            const float residual_term = xsv * wsv[c] * (cross[r][c] - (xcsv * wmv[c]) / 64.0f);
                            v = mu_term + residual_term;
                        }
                        term[(ly + 8 * r) * kPitch + lx + 8 * c] = v;
                    }
                }
            }
            __syncthreads();
            const int live = min(S, G - round * S);
#pragma unroll
            for (int i = 0; i < kSums; ++i) {
                const int p = i * nthreads + tid;
                if (p < TR * TC) {
                    const unsigned char *src = idx_smem + ((p / TC) * kPitch + p % TC) * static_cast<int>(sizeof(acc_t));
                    for (int w = 0; w < live; ++w) acc[i] += *reinterpret_cast<const acc_t *>(src + w * kIdxRegion);
                }
            }
            __syncthreads();
        }
    };
    if (outer != 0) body(std::true_type{});
    else body(std::false_type{});
#pragma unroll
    for (int i = 0; i < kSums; ++i) {
        const int p = i * nthreads + tid;
        const int r = r0 + p / TC, o = o0 + p % TC;
        if (p < TR * TC && r < rows && o < out_f) y[static_cast<int64_t>(r) * out_f + o] = static_cast<float>(acc[i]);
    }
}

template <int BITS, int R, int C, int MAXW>
__global__ void __launch_bounds__(64 * MAXW, MAXW > kIdxMaxWaves ? 1 : R == 1 ? 4 : 3) linear_index_wide_kernel(const IndexArgs p)
{
    __shared__ IndexTables<BITS ? 1 << BITS : 16> tables;
    index_wide_tile<BITS, R, C, kIdxMinWaves, true>(p, blockIdx.y * 8 * R, blockIdx.x * 8 * C, tables, 0);
}

// ---- the packed format on the matrix units ---------------------------------------------------------------------------------
// The table entries are fp32 numbers: over the lowest bit that any of them uses they are integers, and where those have at most 38
// bits the fp64 sum of 64 of them is exact in every order.  The sum over j is then an integer product: the x codes one-hot (2^bits
// bytes of 0 and 1 per j) times the signed base-256 digits of the entries T[.][w_j], one product per digit.  A one-hot operand has
// at most one byte in four, so the products are the 4:2 sparse ones (v_smfmac_i32_32x32x64_i8, twice the dense rate; of the two
// stored bytes of a four only the first is used).  The five int32 sums together are the sum of the table entries, the same double
// that the serial loop ends with, and the group's closed form follows in the same operations: the result's bits stay what they
// are.  Every workgroup looks the table over for its lowest and highest bit.  A table that does not qualify (largest entry more
// than 2^14 times the smallest, subnormals, infinities, NaN: fitted codebooks with a level near zero are like that) runs the loops
// above, 16 rows a tile.
//
// The wide kernel above spends a multiplication, a conversion and an fp64 addition of the vector ALU on every product; here 4 096
// products take five MFMAs of 32 clocks on a pipe of their own.  A wave owns 32 x 32 outputs for all groups, in order.  The digits
// come from a 1 280-byte table in LDS by the w code, 16 bytes a read (2^bits different entries: no bank conflicts, measured); the
// x operand is made in registers, and the fp64 sums lie in LDS between the groups so that three waves fit a SIMD.  What bounds it
// is the LDS: 184 reads of 16 bytes a lane for a wave's group, 160 of them digits; of a launch of 12608 x 1536 -> 384 at 4 bits it
// is busy 64 %, the matrix pipes and the vector ALU (the closed form, 13 instructions per output and group) 47 % each.
// Measured, this kernel against the wide one: 1576 x 384 -> 1536 at 4 / 3 / 2 bits 51 / 44 / 33 us against 103 / 108 / 104, 12608
// rows at 4 bits 309 against 725.  With dense products 82 us; 64 x 32 outputs a wave and the groups dealt over the waves 117.
constexpr int kDigits = 5, kMaxEntryBits = 38;
constexpr int kMfmaTile = 32;                      // a wave's tile is 32 x 32, the workgroup's 32 outputs wide
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));

// The smallest of the lanes' numbers, in a scalar register.
__device__ __forceinline__ int wave_min(int v)
{
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x121, 0xf, 0xf, false));       // row_ror: the minimum of the sixteen lanes
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x122, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x124, 0xf, 0xf, false));
    v = min(v, __builtin_amdgcn_update_dpp(v, v, 0x128, 0xf, 0xf, false));
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <int BITS>
__global__ void __launch_bounds__(64 * kIdxMaxWaves, 3)
linear_index_mfma_kernel(const IndexArgs p)
{
#pragma clang fp contract(off)
    constexpr int L = 1 << BITS, kEntries = L * L, E = 16 / L;                   // E: j's of 16 bytes
    constexpr int kSteps = 16 / E;                                               // 4 E j's each
    __shared__ __attribute__((aligned(16))) signed char s_digits[kDigits * kEntries];        // [digit][w code][x code]
    __shared__ __attribute__((aligned(16))) double s_meta[kIdxMaxWaves][3][kMfmaTile];
    __shared__ IndexTables<L> tables;
    __shared__ int s_low[kIdxMaxWaves], s_high[kIdxMaxWaves];
    extern __shared__ __attribute__((aligned(16))) unsigned char idx_smem[];     // [waves][kIdxRegion]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int nthreads = blockDim.x, S = nthreads >> 6;
    constexpr int kEach = (kEntries + 64 * kIdxMinWaves - 1) / (64 * kIdxMinWaves);
    const int across = (p.out_f + kMfmaTile - 1) / kMfmaTile;                    // workgroups side by side
    const int r0 = blockIdx.x / across * (S * kMfmaTile), ow = blockIdx.x % across * kMfmaTile;
    const int rw = r0 + wave * kMfmaTile;                                        // rows of the wave's tile
    const int G = p.G;

    // Codes of a group: a lane takes j = 32 lh ... + 31 of row lr, and all 64 of output lr.
    // (rows and outputs times groups: 32 bits, checked by the launcher)
    const uint32_t xrow = static_cast<uint32_t>(min(rw + lr, p.rows - 1)) * G, wrow = static_cast<uint32_t>(min(ow + lr, p.out_f - 1)) * G;
    const float *x_meta = lh ? p.xs : p.xc;                                      // (the halves of the wave share the rows' metadata)
    uint32_t xn[BITS], wn[2][BITS];
    float xmn[2], wmn[3];
    auto fetch = [&](int g) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < BITS; ++d) {
            xn[d] = reinterpret_cast<const uint32_t *>(p.xq)[(xrow + g) * (2 * BITS) + lh * BITS + d];
#pragma unroll
            for (int h = 0; h < 2; ++h) wn[h][d] = reinterpret_cast<const uint32_t *>(p.wq)[(wrow + g) * (2 * BITS) + h * BITS + d];
        }
        xmn[0] = x_meta[xrow + g], xmn[1] = p.xcs[xrow + g];
        wmn[0] = p.wc[wrow + g], wmn[1] = p.ws[wrow + g], wmn[2] = p.wcs[wrow + g];
    };
    // The table's entries as integers over 2^low.
    uint32_t entry[kEach];                                                       // (a, b) = (x code, w code) = (i / L, i % L)
    int same = 1, lo = 1 << 20, hi = -(1 << 20);                                           // the bits that any of this thread's use
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int i = tid + k * nthreads;
        entry[k] = i < kEntries ? __float_as_uint(p.table[i]) : 0;
        if (i < kEntries) same &= index_table_entry(p, tables, i, __uint_as_float(entry[k]));
        const int exponent = static_cast<int>((entry[k] >> 23) & 255u);
        if (exponent != 0) lo = min(lo, exponent - 150 + (__ffs(static_cast<int>(entry[k] | 0x800000u)) - 1)), hi = max(hi, exponent - 126);
        if (exponent == 255 || (exponent == 0 && (entry[k] & 0x7fffffu))) hi = 1 << 21;      // infinity, NaN, subnormal: too wide
    }
    lo = wave_min(lo), hi = -wave_min(-hi);
    if (lane == 0) s_low[wave] = lo, s_high[wave] = hi;
    same = __syncthreads_and(same);
    for (int w = 0; w < S; ++w) lo = min(lo, s_low[w]), hi = max(hi, s_high[w]);
    const int low = lo <= hi ? lo : 0;                                           // (else all entries are zero)
    if (hi - low > kMaxEntryBits) {                                              // workgroup-uniform
        const int tiles = across * ((p.rows + 15) / 16), wg = blockIdx.x, shared = tiles - p.singles;
        const int first = wg < p.workers ? wg : shared + wg - p.workers, end = wg < p.workers ? shared : min(first + 1, tiles);
        for (int t = first; t < end; t += p.workers)
            index_wide_tile<BITS, 2, 4, kIdxMinWaves, false>(p, t / across * 16, t % across * 32, tables, same);
        return;
    }
    if (r0 >= p.rows) return;                                                    // (a workgroup that is here for the loops above only)
    fetch(0);
#pragma unroll
    for (int k = 0; k < kEach; ++k) {
        const int i = tid + k * nthreads, exponent = static_cast<int>((entry[k] >> 23) & 255u);
        const int shift = exponent - 150 - low;                                  // (negative: by zero bits of the entry)
        long long v = exponent == 0 ? 0 : static_cast<long long>((entry[k] & 0x7fffffu) | 0x800000u);
        v = shift >= 0 ? v << min(shift, 40) : v >> min(-shift, 23);
        if (entry[k] >> 31) v = -v;
        if (i < kEntries) {
#pragma unroll
            for (int d = 0; d < kDigits; ++d) {
                const signed char digit = static_cast<signed char>(v & 255);
                s_digits[d * kEntries + (i % L) * L + i / L] = digit;
                v = (v - digit) >> 8;
            }
        }
    }
    __syncthreads();
    const int low_s = __builtin_amdgcn_readfirstlane(low);                       // 2^low and 2^(-low - 6), in scalar registers
    if (rw >= p.rows) return;                                                    // (a wave past the last row; there is no barrier below)
    const double unit = __longlong_as_double((1023LL + low_s) << 52), per_unit64 = __longlong_as_double((1017LL - low_s) << 52);

    // Bits from..to (of BITS) of code number q, `up` bits to the left.
    auto code_bits = [](const uint32_t (&w)[BITS], int q, int from, int to, int up) __attribute__((always_inline)) {
        const int bit = q * BITS, d = bit >> 5, sh = bit & 31;
        const uint32_t mask = ((1u << to) - (1u << from)) << up;
        if (sh + BITS > 32) return ((__builtin_amdgcn_alignbit(w[d + 1], w[d], sh)) << up) & mask;
        return (sh >= up ? w[d] >> (sh - up) : w[d] << (up - sh)) & mask;
    };
    // The digits of part k (L bytes) of a 32-byte fragment.
    auto digit_part = [](i32x8_t &f, int k, const signed char *src) __attribute__((always_inline)) {
        if constexpr (L == 16) {
            const int4 v = *reinterpret_cast<const int4 *>(src);
            f[4 * k] = v.x, f[4 * k + 1] = v.y, f[4 * k + 2] = v.z, f[4 * k + 3] = v.w;
        } else if constexpr (L == 8) {
            const int2 v = *reinterpret_cast<const int2 *>(src);
            f[2 * k] = v.x, f[2 * k + 1] = v.y;
        } else {
            f[k] = *reinterpret_cast<const int *>(src);
        }
    };
    // The sums over the groups: lane's outputs v at acc[64 v].
    double *acc = reinterpret_cast<double *>(idx_smem) + wave * 1024 + lane;
    {
        const double b = p.bias && ow + lr < p.out_f ? static_cast<double>(p.bias[ow + lr]) : 0.0;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v * 64] = b;
    }
    double (&meta)[3][kMfmaTile] = s_meta[wave];
#pragma unroll 1
    for (int g = 0; g < G; ++g) {
        uint32_t xk[BITS], wk[2][BITS];
#pragma unroll
        for (int d = 0; d < BITS; ++d) {
            xk[d] = xn[d];
#pragma unroll
            for (int h = 0; h < 2; ++h) {      // lanes of the upper half begin E codes further on
                const uint32_t above = d + 1 < BITS ? wn[h][d + 1] : 0;
                wk[h][d] = lh ? __builtin_amdgcn_alignbit(above, wn[h][d], E * BITS) : wn[h][d];
            }
        }
        // (Multiplying by powers of two commutes with every rounding below: the sums stay in units of 2^low, the scale takes it in.)
        const double wcv = wmn[0], wsv = wmn[1] * unit, wcsv = wmn[2] * per_unit64;
        asm volatile("" ::: "memory");                                           // (the last group's reads of the metadata come first)
        meta[lh][lr] = lh ? static_cast<double>(xmn[0]) : 64.0 * static_cast<double>(xmn[0]);
        meta[2][lr] = xmn[1];
        i32x16_t sum[kDigits];
        int zero = 0;
        asm volatile("" : "+s"(zero));                                           // (of the constant the compiler keeps sixteen in scratch)
#pragma unroll
        for (int d = 0; d < kDigits; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) sum[d][v] = zero;
        // (The reads of a step's digits run under the products before it as far as the registers go: three fragments of eight.)
        i32x4_t xf;
        uint32_t index;
        i32x8_t wf[kDigits];
        auto operands = [&](int t, i32x4_t &a, uint32_t &ix, i32x8_t (&b)[kDigits]) __attribute__((always_inline)) {
            const signed char *src[2 * E];
#pragma unroll
            for (int k = 0; k < 2 * E; ++k) src[k] = s_digits + code_bits(wk[k / E], 2 * E * t + k % E, 0, BITS, BITS);
#pragma unroll
            for (int d = 0; d < kDigits; ++d)
#pragma unroll
                for (int k = 0; k < 2 * E; ++k) digit_part(b[d], k, src[k] + d * kEntries);
            // Stored bytes of the x operand: of the two of a four that the index selects from only the first is used, 1 in the four that
            // the code is in; the index of all its fours is the code's place in one.
            ix = 0;
#pragma unroll
            for (int k = 0; k < 2 * E; ++k) {
                const int q = 2 * E * t + k;
                if constexpr (L == 16) {
                    const uint64_t v = 1ull << code_bits(xk, q, 2, BITS, 2);
                    a[2 * k] = static_cast<int>(v), a[2 * k + 1] = static_cast<int>(v >> 32);
                } else if constexpr (L == 8) {
                    a[k] = static_cast<int>(1u << code_bits(xk, q, 2, BITS, 2));
                } else if (k & 1) {
                    a[k >> 1] = 0x00010001;
                }
                ix |= __umul24(code_bits(xk, q, 0, 2, 0), L == 16 ? 0x1111u : L == 8 ? 0x11u : 0x1u) << (k * L);
            }
        };
#pragma unroll
        for (int t = 0; t < kSteps; ++t) {
            operands(t, xf, index, wf);
#pragma unroll
            for (int d = 0; d < kDigits; ++d)
                sum[d] = __builtin_amdgcn_smfmac_i32_32x32x64_i8(xf, wf[d], sum[d], static_cast<int>(index), 0, 0);
        }
        if (g + 1 < G) fetch(g + 1);                                             // (under the closed form; the products need the registers)
        asm volatile("" ::: "memory");
        // ---- the group's closed form (EXT/arcq_linear_kernel.cu:65-74) ----
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int v = 4 * v4 + e, row = 8 * v4 + 4 * lh + e;
                const int lo = sum[0][v] + sum[1][v] * 256 + sum[2][v] * 65536, hi = sum[3][v] + sum[4][v] * 256;      // |digit sums| <= 2^13
                const double cross = __builtin_fma(static_cast<double>(hi), 16777216.0, static_cast<double>(lo));      // exact
                const double mu_term = meta[0][row] * wcv;
                const double residual_term = meta[1][row] * wsv * (cross - meta[2][row] * wcsv);
                acc[v * 64] += mu_term + residual_term;
            }
        }
    }
    if (ow + lr < p.out_f) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int r = rw + 8 * (v >> 2) + 4 * lh + (v & 3);
            if (r < p.rows) p.y[static_cast<int64_t>(r) * p.out_f + ow + lr] = static_cast<float>(acc[v * 64]);
        }
    }
}

// Waves per workgroup: the count that leaves the fewest of them without a group in the last round, the larger one of equals
// (384 -> 1536, six groups, 12608 rows, wide kernel: three waves 744, four waves 832 us).
inline int index_waves(int G)
{
    int S = kIdxMaxWaves;
    for (int s = kIdxMaxWaves - 1; s >= kIdxMinWaves; --s)
        if ((G + s - 1) / s * s < (G + S - 1) / S * S) S = s;
    return S;
}

// The host does not see the table, so the launch serves both cases.  Waves per workgroup as above (1576 x 384 -> 1536 51.0 us with
// three, 51.7 with four: the matrix-unit tiles are a wave's own), but four where three would put more wave tiles on the busiest SIMD
// (workgroups are dealt whole: 5721 x 1344 -> 352 at 2 bits 81 us with three, 66 with four; 9303 x 1088 -> 224 94 and 78).
//
// Tables that do not qualify: where the workgroups above would leave compute units idle, more are launched for the 16-row tiles of the
// loops, as many as are resident at once; a table that qualifies sends them home after the look at it (512 x 384 -> 1024 24.5 us with
// and without them).  Four waves: from one resident set on that set shares the tiles and every workgroup behind it takes one of the
// last ones, which evens out the end; from four tiles for each on there are a third more for that (2343 x 448 -> 960 124 -> 113 us,
// 3192 x 1408 -> 736 358 -> 324; 6170 x 1472 -> 1408, dealt to all 2156 workgroups alike, 1326 -> 1210).  Three waves, of which not
// quite four workgroups fit a compute unit: the tiles are dealt to fifteen sixteenths of a resident set, from three sets on to all
// (12608 x 384 -> 1536: to all 761 us, the four waves' rule 894; 5000 x 576 -> 768 273 and 285).
// Against the wide kernel alone, at 44 sizes of 512 .. 12608 rows and 2 .. 24 groups: with computed entries 0.96 of its speed in the
// mean (512 x 384 -> 1024 27.4 / 26.8 us, 1576 x 384 -> 1536 111 / 105, 12608 x 384 -> 1536 758 / 710; at worst, where two rounds are
// not full, 5000 x 576 -> 768 273 / 218), with gathered ones 0.99 (at worst, nine groups on four waves, 10800 x 576 -> 1056
// 1620 / 1350).  (Eight tiles in turn per 128-row workgroup: 512 rows 100 us, 1576 164, 12608 936.)
template <int BITS>
void launch_index_mfma(const IndexArgs &a, hipStream_t stream)
{
    const int across = (a.out_f + kMfmaTile - 1) / kMfmaTile;
    auto workgroups = [&](int waves) { return across * ((a.rows + waves * kMfmaTile - 1) / (waves * kMfmaTile)); };
    auto busiest_simd = [&](int waves) { return ((workgroups(waves) + device_cus() - 1) / device_cus() * waves + 3) / 4; };
    int S = index_waves(a.G);
    if (busiest_simd(S) > busiest_simd(kIdxMaxWaves)) S = kIdxMaxWaves;
    const int resident = 4 * kIdxMinWaves / S * device_cus(), tiles = across * ((a.rows + 15) / 16), own = workgroups(S);
    const int grid = max(own, min(tiles, S == kIdxMaxWaves && tiles >= 4 * resident ? resident + resident / 3 : resident));
    IndexArgs b = a;
    b.workers = S == kIdxMaxWaves ? min(grid, resident) : own <= resident || own >= 3 * resident ? grid : resident - resident / 16;
    b.singles = S == kIdxMaxWaves ? grid - b.workers : 0;
    hipLaunchKernelGGL((linear_index_mfma_kernel<BITS>), dim3(grid), dim3(64 * S), S * kIdxRegion, stream, b);
}

template <int BITS, int R, int C, int MAXW>
void launch_index_wide(const IndexArgs &a, hipStream_t stream)
{
    // Of up to sixteen waves the fewest for the fewest rounds.
    int S = index_waves(a.G);
    if constexpr (MAXW > kIdxMaxWaves) {
        const int rounds = (a.G + MAXW - 1) / MAXW;
        S = (a.G + rounds - 1) / rounds;
        allow_dynamic_lds<linear_index_wide_kernel<BITS, R, C, MAXW>>(MAXW * kIdxRegion);
    }
    hipLaunchKernelGGL((linear_index_wide_kernel<BITS, R, C, MAXW>), dim3((a.out_f + 8 * C - 1) / (8 * C), (a.rows + 8 * R - 1) / (8 * R)), dim3(64 * S),
                       S * kIdxRegion, stream, a);
}
// Four outputs and two rows per lane; one row where that leaves at most 1024 workgroups (four per CU), whose duration is
// one wave's (197 x 768 -> 768, 600 of them: 30.6 against 34.2 us; 394 x 768 -> 768: 42.4 against 42.9, byte codes 40.6
// against 34.5).  Four rows spill nothing but leave two waves per SIMD: 1576 x 384 -> 1536 131 us against 121.
template <int BITS>
void launch_index(const IndexArgs &a, hipStream_t stream)
{
    const int64_t small_tiles = static_cast<int64_t>((a.rows + 7) / 8) * ((a.out_f + 31) / 32);
    // The matrix units from 1024 half tiles of 16 x 32 on (two wave tiles of 32 x 32 for every compute unit), whatever the number of
    // groups: 788 x 768 -> 768 (1200 of them) 45 against 57 us, 394 x 1536 -> 1536 (1200) 83.5 / 106; below, a wave's chain over all
    // groups is what the launch takes: 394 x 768 -> 768 (600) 45.2 against 34.6 us, 197 x 192 -> 768 (312) 16.1 / 10.1.  Half tiles,
    // because padding counts: 16 x 384 -> 16416 (513) 24.6 / 24.7, 8 rows 25 / 16, 48 x 384 -> 8225 (774) 29 / 26.5, 24 x 384 -> 16416
    // (1026) 25 / 35, 64 x 384 -> 8225 (1032) 29.5 / 34.6, 16416 x 384 -> 8 (1026) 24 / 32.6.
    if constexpr (BITS != 0) {
        const int64_t halves = static_cast<int64_t>((a.rows + 15) / 16) * ((a.out_f + kMfmaTile - 1) / kMfmaTile);
        if (halves >= 4 * device_cus() && halves < (int64_t(1) << 24) && static_cast<int64_t>(a.rows > a.out_f ? a.rows : a.out_f) * a.G * 2 * BITS < (int64_t(1) << 31))
            return launch_index_mfma<BITS>(a, stream);
    }
    // No more workgroups than compute units: up to sixteen waves each, i.e. as few rounds of groups as possible.
    if (small_tiles <= device_cus() && a.G > kIdxMaxWaves) launch_index_wide<BITS, 1, 4, 16>(a, stream);
    else if (small_tiles <= 1024) launch_index_wide<BITS, 1, 4, kIdxMaxWaves>(a, stream);
    else launch_index_wide<BITS, 2, 4, kIdxMaxWaves>(a, stream);
}

// Launches of at most this many 16 x 64 tiles give every thread one output instead of four.
constexpr int kSmallTiles = 512;
static size_t tile_table_bytes(int levels) { return static_cast<size_t>(levels) * levels * sizeof(float); }

static int check_common(const char *fn, int64_t rows, int64_t out_f, int64_t in_f, int gs, int levels)
{
    if (rows < 0 || out_f < 0 || in_f < 0 || gs <= 0) return fail(ARCQ_ERR_SHAPE, "%s: bad sizes", fn);
    if (in_f % gs != 0) return fail(ARCQ_ERR_GROUP, "%s: in_features must be divisible by group_size", fn);
    // (the table is held in LDS: 128 x 128 floats are 64 KB)
    if (levels < 1 || levels > 128) return fail(ARCQ_ERR_SHAPE, "%s: product_table must be [levels, levels] with 1 <= levels <= 128 (got %d)", fn, levels);
    if ((out_f + kIdxTile - 1) / kIdxTile > 0x7fffffff || (rows + kIdxTile - 1) / kIdxTile > 65535)
        return fail(ARCQ_ERR_SHAPE, "%s: too many rows or outputs", fn);
    return ARCQ_OK;
}

}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_linear_forward_packed(const uint8_t *packed_x, const float *x_center, const float *x_scale,
                                        const float *x_code_sum,
                                        const uint8_t *packed_w, const float *w_center, const float *w_scale,
                                        const float *w_code_sum,
                                        const float *product_table, const float *bias, float *y,
                                        int64_t rows, int64_t out_features, int64_t in_features,
                                        int bits, int group_size, int levels, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_linear_forward_packed: bits must be 2, 3, or 4");
    int rc = check_common("arcq_linear_forward_packed", rows, out_features, in_features, group_size, levels);
    if (rc != ARCQ_OK) return rc;
    if (levels < (1 << bits))
        return fail(ARCQ_ERR_SHAPE, "arcq_linear_forward_packed: product_table has %d levels, %d-bit codes need %d",
                    levels, bits, 1 << bits);
    if (rows * out_features == 0) return ARCQ_OK;
    if (!y || !product_table) return fail(ARCQ_ERR_NULL, "arcq_linear_forward_packed: NULL tensor pointer");
    if (in_features > 0 && (!packed_x || !x_center || !x_scale || !x_code_sum || !packed_w || !w_center || !w_scale || !w_code_sum))
        return fail(ARCQ_ERR_NULL, "arcq_linear_forward_packed: NULL tensor pointer");
    if (group_size == 64 && in_features > 0 && (rows + kTileRows - 1) / kTileRows <= 65535 && aligned(packed_x, 4) &&
        aligned(packed_w, 4)) {
        dim3 tgrid(static_cast<unsigned>((out_features + kTileOuts - 1) / kTileOuts),
                   static_cast<unsigned>((rows + kTileRows - 1) / kTileRows));
        const bool small = static_cast<int64_t>(tgrid.x) * tgrid.y <= kSmallTiles;
#define ARCQ_LAUNCH_TILE(B, O)                                                                                           \
    do {                                                                                                                  \
        allow_dynamic_lds<linear_index_tile_kernel<B, O>>(64 * 1024);                                                     \
        hipLaunchKernelGGL((linear_index_tile_kernel<B, O>), tgrid, dim3(1024 / O), tile_table_bytes(levels),              \
                           static_cast<hipStream_t>(stream), packed_x, x_center, x_scale, x_code_sum, packed_w, w_center, \
                           w_scale, w_code_sum, product_table, bias, y, rows, out_features, in_features, levels);         \
    } while (0)
        if (bits == 4) { if (small) ARCQ_LAUNCH_TILE(4, 1); else ARCQ_LAUNCH_TILE(4, 4); }
        else if (bits == 3) { if (small) ARCQ_LAUNCH_TILE(3, 1); else ARCQ_LAUNCH_TILE(3, 4); }
        else { if (small) ARCQ_LAUNCH_TILE(2, 1); else ARCQ_LAUNCH_TILE(2, 4); }
#undef ARCQ_LAUNCH_TILE
        return launch_status("arcq_linear_forward_packed");
    }
    // Any other group size: one thread per output, codes extracted from global memory (slow, no layout assumptions).
    dim3 grid(static_cast<unsigned>((out_features + kIdxTile - 1) / kIdxTile),
              static_cast<unsigned>((rows + kIdxTile - 1) / kIdxTile));
    allow_dynamic_lds<linear_index_packed_kernel>(64 * 1024);
    hipLaunchKernelGGL(linear_index_packed_kernel, grid, dim3(256), levels * levels * sizeof(float),
                       static_cast<hipStream_t>(stream), packed_x, x_center, x_scale, x_code_sum, packed_w, w_center,
                       w_scale, w_code_sum, product_table, bias, y, rows, out_features, in_features, bits, group_size,
                       levels);
    return launch_status("arcq_linear_forward_packed");
}

ARCQ_API int arcq_linear_forward_u8(const uint8_t *x_codes, const float *x_center, const float *x_scale,
                                    const float *x_code_sum,
                                    const uint8_t *w_codes, const float *w_center, const float *w_scale,
                                    const float *w_code_sum,
                                    const float *product_table, const float *bias, float *y,
                                    int64_t rows, int64_t out_features, int64_t in_features,
                                    int group_size, int levels, void *stream)
{
    int rc = check_common("arcq_linear_forward_u8", rows, out_features, in_features, group_size, levels);
    if (rc != ARCQ_OK) return rc;
    if (rows * out_features == 0) return ARCQ_OK;
    if (!y || !product_table) return fail(ARCQ_ERR_NULL, "arcq_linear_forward_u8: NULL tensor pointer");
    if (in_features > 0 && (!x_codes || !x_center || !x_scale || !x_code_sum || !w_codes || !w_center || !w_scale || !w_code_sum))
        return fail(ARCQ_ERR_NULL, "arcq_linear_forward_u8: NULL tensor pointer");
    if (group_size == 64 && in_features > 0 && (rows + kTileRows - 1) / kTileRows <= 65535 && aligned(x_codes, 4) &&
        aligned(w_codes, 16)) {
        dim3 tgrid(static_cast<unsigned>((out_features + kTileOuts - 1) / kTileOuts),
                   static_cast<unsigned>((rows + kTileRows - 1) / kTileRows));
        if (static_cast<int64_t>(tgrid.x) * tgrid.y <= kSmallTiles) {
            allow_dynamic_lds<linear_index_tile_kernel<0, 1>>(64 * 1024);
            hipLaunchKernelGGL((linear_index_tile_kernel<0, 1>), tgrid, dim3(1024), tile_table_bytes(levels),
                               static_cast<hipStream_t>(stream), x_codes, x_center, x_scale, x_code_sum, w_codes, w_center,
                               w_scale, w_code_sum, product_table, bias, y, rows, out_features, in_features, levels);
        } else {
            allow_dynamic_lds<linear_index_tile_kernel<0, 4>>(64 * 1024);
            hipLaunchKernelGGL((linear_index_tile_kernel<0, 4>), tgrid, dim3(256), tile_table_bytes(levels),
                               static_cast<hipStream_t>(stream), x_codes, x_center, x_scale, x_code_sum, w_codes, w_center,
                               w_scale, w_code_sum, product_table, bias, y, rows, out_features, in_features, levels);
        }
        return launch_status("arcq_linear_forward_u8");
    }
    dim3 grid(static_cast<unsigned>((out_features + kIdxTile - 1) / kIdxTile),
              static_cast<unsigned>((rows + kIdxTile - 1) / kIdxTile));
    allow_dynamic_lds<linear_index_u8_kernel>(64 * 1024);
    hipLaunchKernelGGL(linear_index_u8_kernel, grid, dim3(256), levels * levels * sizeof(float),
                       static_cast<hipStream_t>(stream), x_codes, x_center, x_scale, x_code_sum, w_codes, w_center,
                       w_scale, w_code_sum, product_table, bias, y, rows, out_features, in_features, group_size, levels);
    return launch_status("arcq_linear_forward_u8");
}

ARCQ_API int arcq_linear_index(const arcq_linear_index_args *a, void *stream)
{
    if (!a) return fail(ARCQ_ERR_NULL, "arcq_linear_index: args must not be NULL");
    if (a->bits != 0 && !bits_ok(a->bits)) return fail(ARCQ_ERR_BITS, "arcq_linear_index: bits must be 2, 3, or 4 (or 0 for byte codes)");
    const bool wide = a->group_size == 64 && a->in_features > 0 && a->in_features % 64 == 0 && a->levels >= 1 && a->a_codebook && a->w_codebook &&
                      (a->bits ? a->levels == (1 << a->bits) : a->levels <= 16) && a->rows > 0 && a->out_features > 0 &&
                      a->rows < (1 << 19) && a->out_features < (1 << 28) && a->x_codes && a->x_center && a->x_scale && a->x_code_sum &&
                      a->w_codes && a->w_center && a->w_scale && a->w_code_sum && a->product_table && a->y && aligned(a->x_codes, 8) &&
                      aligned(a->w_codes, 8);
    if (!wide) {           // anything else, and what is wrong: the entry points that take no codebooks
        if (a->bits)
            return arcq_linear_forward_packed(a->x_codes, a->x_center, a->x_scale, a->x_code_sum, a->w_codes, a->w_center, a->w_scale,
                                              a->w_code_sum, a->product_table, a->bias, a->y, a->rows, a->out_features, a->in_features,
                                              a->bits, a->group_size, a->levels, stream);
        return arcq_linear_forward_u8(a->x_codes, a->x_center, a->x_scale, a->x_code_sum, a->w_codes, a->w_center, a->w_scale, a->w_code_sum,
                                      a->product_table, a->bias, a->y, a->rows, a->out_features, a->in_features, a->group_size, a->levels,
                                      stream);
    }
    const IndexArgs g{a->x_codes, a->x_center, a->x_scale, a->x_code_sum, a->w_codes, a->w_center, a->w_scale, a->w_code_sum, a->product_table,
                      a->a_codebook, a->w_codebook, a->bias, a->y, static_cast<int>(a->rows), static_cast<int>(a->out_features),
                      static_cast<int>(a->in_features / 64), a->levels, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->bits == 4) launch_index<4>(g, st);
    else if (a->bits == 3) launch_index<3>(g, st);
    else if (a->bits == 2) launch_index<2>(g, st);
    else launch_index<0>(g, st);
    return launch_status("arcq_linear_index");
}
