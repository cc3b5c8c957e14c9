// Softmax attention of a ViT block, placed between the packed qkv and proj layers so that neither needs a reshaping
// kernel around it: it reads the qkv layer's output as it is and writes the proj layer's input as it is.
//
//   qkv [B, n, 3, H, 64] fp16  (= the qkv layer's y, [B*n, 3*H*64] row-major: q, k, v of head h at columns
//                               (0|1|2)*H*64 + h*64 ...)
//   out [B, n, H*64]     fp16  (= the proj layer's x):  out[b, i, h*64 + j] = sum_k softmax_k(q_i . k_k * scale) v_k[j]
//
// No counterpart in the reference's packed path (its models run timm's attention through torch); part of the
// whole-block fusion around the packed linears: at batch 1 the library attention plus the two copies that reshape
// its operands take as long as two packed layers.
//
// One workgroup per (batch, head), or where these are few one per part of a head: wave w owns the 32 queries of tile w, or of tile
// parts * w + part, and the waves without a tile only load (n <= 256 tokens: at most eight waves).  K of
// the head sits in LDS row-major, V transposed, both zero-padded to whole 32-key blocks.  Scores: S^T = K Q^T on
// v_mfma_f32_32x32x16_f16 with K as the first operand, so that a lane (query q = lane % 32, half h = lane / 32) ends
// up holding, of every 32-key block, the 16 keys 8 t + 4 h + c (t, c = 0..3) of its own query: the row maximum and sum
// are in-lane reductions plus one exchange with lane ^ 32, and -- since the contraction index of the second product
// may be enumerated in any order as long as both operands use the same one -- eight consecutive accumulator registers,
// rounded to fp16, ARE the second operand of O^T = V^T P^T for the keys {16 s + 4 h + c, 16 s + 8 + 4 h + c}; the
// matching eight values of V^T are two 8-byte LDS reads.  fp32 scores, softmax and accumulation; P rounded to fp16;
// normalisation by the row sum at the end.  Beyond 128 keys the keys go in two chunks with a running maximum and sum.
#include "arcq_act_quant_core.h"
#include "arcq_gemm.h"

#include <algorithm>

namespace arcq {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kHeadDim = 64;
constexpr int kKPitch = kHeadDim * 2 + 16;          // bytes per key row of K in LDS

// NKB = 32-key blocks (= 32-query tiles = waves): ceil(n / 32).
// NQ = 0, or the bits of the proj layer's activation quantizer: `out` then receives that layer's x_hat (stage 1 of the
// rounded output; a head's 64 dims are one quantization group) in the 32-row block layout of the [B n, C] tensor instead of
// the output.  A wave's 32 x 64 outputs go through its own 32 rows of K in LDS (all waves are done with it) into the
// lane-pair routine of the GEMM epilogues.
// F8: that operand as FP8 (rows padded to 128 values).
// SPLIT: a head has gridDim.z workgroups.  (A template: the two registers that it takes cost 5 % at 256 images of 16 heads.)
// FEW: the last key block holds at most eight keys (197 or 101 tokens: five).  The other 24 would get scores of minus infinity and
// probabilities of zero: no maximum, no exponentials, no second half of the product.  197 tokens (the vector instructions bound it, a
// tenth of them are gone): 64 images of 6 heads 17.8 -> 16.9 us, of 12 28.7 -> 27.9, 256 of 16 with proj's stage 1 137 -> 133, one of 6
// 7.1 -> 6.9.  A template: as a branch on the number of keys it spills 13 to 69 registers.
template <int NKB, int NQ, bool F8, bool SPLIT, bool FEW>
__global__ void __launch_bounds__(64 * NKB) __attribute__((amdgpu_waves_per_eu(SPLIT ? 2 : 4)))     // two workgroups of up to 8 waves on a CU, or one
attention_kernel(const __half *__restrict__ qkv, __half *__restrict__ out, int n, int H, float scale,
                 const float *__restrict__ nq_thr, const float *__restrict__ nq_cb, int total_rows)
{
    constexpr int kKeys = 32 * NKB;
    // bytes per dim row of V^T in LDS: the row stride in dwords is 2 mod 4, which spreads both the transposing writes
    // (rows 8 apart, 4-byte) and the product's reads (32 consecutive rows, 8-byte) over the banks
    constexpr int kVPitch = kKeys * 2 + 8;
    constexpr int CH = NKB <= 4 ? 4 : NKB == 6 ? 2 : 3;   // key blocks whose scores are live at a time (no spills at 128 registers)
    constexpr int NCH = (NKB + CH - 1) / CH;
    __shared__ __attribute__((aligned(16))) unsigned char ks[kKeys * kKPitch];
    __shared__ __attribute__((aligned(16))) unsigned char vt[kHeadDim * kVPitch];
    __shared__ __attribute__((aligned(16))) unsigned char nq_lds[NQ ? next_quant_lds_bytes() : 16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int h = blockIdx.x, b = blockIdx.y;
    const int C = H * kHeadDim;
    const int64_t row0 = static_cast<int64_t>(b) * n;           // first token row of this image
    const __half *base = qkv + h * kHeadDim;                    // + (row * 3 + which) * C

    // ---- K row-major and V transposed into LDS (keys past n as zeros).  16 NKB key pairs x 8 pieces of 8 dims =
    //      exactly two items per thread; all eight loads are in flight before the first LDS write ----
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    QuantParams nq_params{};
    if constexpr (NQ != 0) {                                   // (the last wave has the fewest queries)
        if (wave == NKB - 1) nq_params = load_quant_params<NQ>(nq_thr, nq_cb, lane);
    }
    u32x4_t kreg[2][2], vreg[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int p = tid + i * 64 * NKB, kp = p >> 3, piece = p & 7;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int key = 2 * kp + j;
            const __half *src = base + ((row0 + min(key, n - 1)) * 3 + 1) * C + piece * 8;
            kreg[i][j] = key < n ? *reinterpret_cast<const u32x4_t *>(src) : zero4;
            vreg[i][j] = key < n ? *reinterpret_cast<const u32x4_t *>(src + C) : zero4;
        }
    }
    if constexpr (NQ != 0 && !SPLIT) {                         // while K and V are on their way
        if (wave == NKB - 1) next_quant_setup<NQ>(nq_params, nq_lds, lane);
    }
    // ---- this wave's queries: lane (q, half) holds Q[q][16 kk + 8 half ... + 7] for kk = 0..3 ----
    const int tile = SPLIT ? wave * gridDim.z + blockIdx.z : wave;      // (parts of a head take its query tiles in turn)
    const bool busy = !SPLIT || tile < NKB;
    const int q = tile * 32 + lr;
    u32x4_t qf[4];
    {
        const __half *src = base + (row0 + min(q, n - 1)) * 3 * C + 8 * lh;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) qf[kk] = q < n ? *reinterpret_cast<const u32x4_t *>(src + 16 * kk) : zero4;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int p = tid + i * 64 * NKB, kp = p >> 3, piece = p & 7;
#pragma unroll
        for (int j = 0; j < 2; ++j)
            *reinterpret_cast<u32x4_t *>(ks + (2 * kp + j) * kKPitch + piece * 16) = kreg[i][j];
#pragma unroll
        for (int e = 0; e < 8; ++e) {       // dim piece*8 + e of the two keys as one dword
            const uint32_t a = vreg[i][0][e >> 1], c = vreg[i][1][e >> 1];
            const uint32_t pair = (e & 1) ? ((a >> 16) | (c & 0xffff0000u)) : ((a & 0xffffu) | (c << 16));
            *reinterpret_cast<uint32_t *>(vt + (piece * 8 + e) * kVPitch + kp * 4) = pair;
        }
    }
    __syncthreads();

    if (NQ == 0 && !busy) return;
    if constexpr (NQ != 0 && SPLIT) {                          // (under the others' product: that wave has no tile in a part)
        if (wave == NKB - 1) next_quant_setup<NQ>(nq_params, nq_lds, lane);
    }
    // Keys in chunks of CH blocks with a running maximum and sum (the scores of one chunk are live at a time, which
    // keeps the wave at half the registers and two workgroups on a CU); one chunk is the plain two-pass softmax.
    const float ninf = -__builtin_inff();
    const float c2 = scale * 1.44269504088896341f;      // exp(scale x) = exp2(c2 x)
    float m = ninf, l = 0.0f;
    float16_t oacc[2];      // oacc[jb][v]: dim jb*32 + 8 (v / 4) + 4 lh + v % 4 of this lane's query
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
        for (int v = 0; v < 16; ++v) oacc[jb][v] = 0.0f;
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
        if (NQ != 0 && !busy) break;                            // (the wave has a barrier left)
        constexpr int kLast = NKB - CH * (NCH - 1);
        const int nb = ch == NCH - 1 ? kLast : CH;          // constant after unrolling
        if (ch > 0) __builtin_amdgcn_sched_barrier(0);      // keep the next chunk's scores out of this one's live range
        // ---- scores: acc[i][v] = q . k for key (ch*CH + i)*32 + 8 (v / 4) + 4 lh + v % 4 ----
        float16_t acc[CH];
        float cm = ninf;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (i >= nb) continue;
            const int kb = ch * CH + i;
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const half8_t kf = *reinterpret_cast<const half8_t *>(ks + (kb * 32 + lr) * kKPitch + (16 * kk + 8 * lh) * 2);
                half8_t qv;
                __builtin_memcpy(&qv, &qf[kk], 16);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qv, acc[i], 0, 0, 0);
            }
            // (raw scores: the scale is positive, so it commutes with the maximum and is applied inside the exponential;
            // only the last key block can hold keys past n)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                if (FEW && kb == NKB - 1 && v >= 4) break;
                if (kb == NKB - 1) {
                    const int key = kb * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
                    acc[i][v] = key < n ? acc[i][v] : ninf;
                }
                cm = fmaxf(cm, acc[i][v]);
            }
        }
        cm = fmaxf(cm, __shfl_xor(cm, 32));
        const float m_new = fmaxf(m, cm);       // finite: every chunk holds at least one key < n
        if (ch > 0) {                           // rescale what the earlier chunks left (exp(-inf) never occurs here)
            const float alpha = __builtin_amdgcn_exp2f((m - m_new) * c2);
            l *= alpha;
#pragma unroll
            for (int jb = 0; jb < 2; ++jb)
#pragma unroll
                for (int v = 0; v < 16; ++v) oacc[jb][v] *= alpha;
        }
        m = m_new;
        const float mc = -m * c2;
        // ---- probabilities (this lane's share of the row sum; the two halves are added at the end) and O^T += V^T P^T ----
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            if (i >= nb) continue;
            const int kb = ch * CH + i;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                if (FEW && kb == NKB - 1 && v >= 4) {
                    acc[i][v] = 0.0f;
                    continue;
                }
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(acc[i][v], c2, mc));      // exp(scale (s - m))
                acc[i][v] = p;
                l += p;
            }
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (FEW && kb == NKB - 1 && s == 1) break;
                half8_t pf;
#pragma unroll
                for (int e = 0; e < 8; ++e) pf[e] = static_cast<_Float16>(acc[i][8 * s + e]);
#pragma unroll
                for (int jb = 0; jb < 2; ++jb) {
                    const unsigned char *vrow = vt + (jb * 32 + lr) * kVPitch + (kb * 32 + 16 * s + 4 * lh) * 2;
                    const u32x2_t lo = *reinterpret_cast<const u32x2_t *>(vrow);
                    const u32x2_t hi = *reinterpret_cast<const u32x2_t *>(vrow + 16);
                    half8_t vf;
                    __builtin_memcpy(&vf, &lo, 8);
                    __builtin_memcpy(reinterpret_cast<char *>(&vf) + 8, &hi, 8);
                    oacc[jb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf, oacc[jb], 0, 0, 0);
                }
            }
        }
    }
    l += __shfl_xor(l, 32);
    if constexpr (NQ != 0) {
        __syncthreads();                                     // everyone is done with K
        unsigned char *stage = ks + wave * 32 * kKPitch;
        const float inv = 1.0f / l;
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (!busy) break;
                const __half2 a = __floats2half2_rn(oacc[jb][4 * t] * inv, oacc[jb][4 * t + 1] * inv);
                const __half2 c = __floats2half2_rn(oacc[jb][4 * t + 2] * inv, oacc[jb][4 * t + 3] * inv);
                u32x2_t pk;
                pk[0] = *reinterpret_cast<const uint32_t *>(&a);
                pk[1] = *reinterpret_cast<const uint32_t *>(&c);
                *reinterpret_cast<u32x2_t *>(stage + lr * kKPitch + (jb * 32 + 8 * t + 4 * lh) * 2) = pk;
            }
        const int parts = SPLIT ? gridDim.z : 1;
        if (SPLIT && 4 * ((NKB + parts - 1) / parts) <= NKB) {
            // Few waves have a tile, but all of them quantize: eight lanes a row (FP8: four), one 16-byte piece a lane.  With one
            // tile to four or more waves that beats two lanes a row on the waves that have one at every size measured (4 to 8 waves,
            // one tile: 0.86 .. 0.95 of its time; 8 waves, two tiles: 0.88); with fewer it does not (2 and 3 waves: 1.05 .. 1.09;
            // two tiles to 3 .. 7 waves: 1.00 .. 1.24; three or four tiles: 0.97 .. 1.15), but for FP8 with two tiles to 7 waves (0.93).
            constexpr int V = F8 ? 16 : 8, LANES = 64 / V, ROWS = 64 / LANES;
            __syncthreads();
            const int part = blockIdx.z, tiles = (NKB - part + parts - 1) / parts;
            for (int job = wave; job < tiles * (32 / ROWS); job += NKB) {
                const int at = job * ROWS + lane / LANES, piece = lane % LANES;       // row of the part, piece of the row
                float v[V];
#pragma unroll
                for (int i = 0; i < V / 8; ++i) {
                    const u32x4_t w = *reinterpret_cast<const u32x4_t *>(ks + at * kKPitch + (piece * (V / 8) + i) * 16);
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        v[8 * i + 2 * d] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] & 0xffffu)));
                        v[8 * i + 2 * d + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] >> 16)));
                    }
                }
                next_quant_lanes<NQ>(nq_lds, v, lane, 1.0e-6f);
                const int qr = ((at >> 5) * parts + part) * 32 + (at & 31);
                if (qr < n) {
                    const int64_t row = row0 + qr;
                    const int blk = static_cast<int>(row >> 5), nrows = min(32, total_rows - blk * 32);
                    const int row_bytes = F8 ? (C + 127) / 128 * 128 : C * 2;
                    char *dst = reinterpret_cast<char *>(out) + static_cast<int64_t>(blk) * 32 * row_bytes +
                                (static_cast<int64_t>(h * LANES + piece) * nrows + (row & 31)) * 16;
                    uint32_t o[4];
                    if constexpr (F8) {
                        float lo[8], hi[8];
#pragma unroll
                        for (int e = 0; e < 8; ++e) lo[e] = v[e], hi[e] = v[V - 8 + e];
                        to_fp8x8(lo, o[0], o[1]);
                        to_fp8x8(hi, o[2], o[3]);
                    } else {
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            const __half2 pr = __floats2half2_rn(v[2 * d], v[2 * d + 1]);
                            o[d] = *reinterpret_cast<const uint32_t *>(&pr);
                        }
                    }
                    store_writethrough16(dst, o[0], o[1], o[2], o[3]);
                    if (F8 && h == H - 1 && (H & 1) != 0) store_writethrough16(dst + LANES * nrows * 16, 0, 0, 0, 0);
                }
            }
            return;
        }
        if (!busy) return;
        __builtin_amdgcn_wave_barrier();
        // This lane's row of the chunk (rows past the image's last query: zero scores of zero queries, not stored).
        const int qr = tile * 32 + (lane >> 1);
        const int64_t row = row0 + qr;
        const int blk = static_cast<int>(row >> 5);
        const int nrows = min(32, total_rows - blk * 32);
        const int row_bytes = F8 ? (C + 127) / 128 * 128 : C * 2;
        char *dst = reinterpret_cast<char *>(out) + static_cast<int64_t>(blk) * 32 * row_bytes + (static_cast<int64_t>(h) * (F8 ? 4 : 8) * nrows + (row & 31)) * 16;
        next_quant_rows<NQ, F8>(nq_lds, stage, kKPitch, lane, false, 1.0e-6f, dst, nrows, qr < n, F8 && h == H - 1 && (H & 1) != 0);
        return;
    }
    // ---- normalise, round, store: each lane 4 runs of 4 consecutive dims per 32-dim block ----
    if (q < n) {
        const float inv = 1.0f / l;
        __half *dst = out + (row0 + q) * C + h * kHeadDim;
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const __half2 a = __floats2half2_rn(oacc[jb][4 * t] * inv, oacc[jb][4 * t + 1] * inv);
                const __half2 c = __floats2half2_rn(oacc[jb][4 * t + 2] * inv, oacc[jb][4 * t + 3] * inv);
                u32x2_t pk;
                pk[0] = *reinterpret_cast<const uint32_t *>(&a);
                pk[1] = *reinterpret_cast<const uint32_t *>(&c);
                *reinterpret_cast<u32x2_t *>(dst + jb * 32 + 8 * t + 4 * lh) = pk;
            }
    }
}

template <int NKB, int NQ, bool F8>
void launch_attention(const void *qkv, void *out, int B, int n, int H, float scale, const float *thr, const float *cb, hipStream_t stream)
{
    // Parts of a head: as many as the compute units take, so that the waves that share a SIMD in a workgroup of a whole head have one
    // each, the tables are built under the product and (one tile a part) all waves share the consumer's stage 1.  197 tokens of 6
    // heads with that stage 1: 9.5 us in one part, 6.5 in seven; 16 images 9.9 and 7.7 in two parts.
    const int64_t heads = static_cast<int64_t>(B) * H;
    const int parts = static_cast<int>(std::min<int64_t>(NKB, std::max<int64_t>(1, device_cus() / heads)));
    const bool few = n - 32 * (NKB - 1) <= 8;
    auto kernel = NKB > 1 && parts > 1 ? (few ? attention_kernel<NKB, NQ, F8, (NKB > 1), true> : attention_kernel<NKB, NQ, F8, (NKB > 1), false>)
                                       : (few ? attention_kernel<NKB, NQ, F8, false, true> : attention_kernel<NKB, NQ, F8, false, false>);
    hipLaunchKernelGGL(kernel, dim3(H, B, parts), dim3(64 * NKB), 0, stream, static_cast<const __half *>(qkv),
                       static_cast<__half *>(out), n, H, scale, thr, cb, B * n);
}

template <int NQ, bool F8 = false>
void launch_attention_n(const void *qkv, void *out, int B, int n, int H, float scale, const float *thr, const float *cb, hipStream_t st)
{
    switch ((n + 31) / 32) {
    case 1: launch_attention<1, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 2: launch_attention<2, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 3: launch_attention<3, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 4: launch_attention<4, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 5: launch_attention<5, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 6: launch_attention<6, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    case 7: launch_attention<7, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    default: launch_attention<8, NQ, F8>(qkv, out, B, n, H, scale, thr, cb, st); break;
    }
}

int attention_checked(const char *fn, const void *qkv, void *out, int64_t B, int64_t n, int64_t H, int64_t head_dim, float scale,
                      int nq_bits, const float *thr, const float *cb, void *stream, bool fp8 = false)
{
    if (B < 0 || n < 0 || H < 0) return fail(ARCQ_ERR_SHAPE, "%s: negative size", fn);
    if (!(scale > 0.0f)) return fail(ARCQ_ERR_UNSUPPORTED, "%s: scale must be positive", fn);
    if (head_dim != kHeadDim) return fail(ARCQ_ERR_UNSUPPORTED, "%s: head_dim must be 64 (got %lld)", fn, static_cast<long long>(head_dim));
    if (n > 256) return fail(ARCQ_ERR_UNSUPPORTED, "%s: at most 256 tokens (got %lld)", fn, static_cast<long long>(n));
    if (B * n * H == 0) return ARCQ_OK;
    if (!qkv || !out || (nq_bits && (!thr || !cb))) return fail(ARCQ_ERR_NULL, "%s: NULL tensor pointer", fn);
    if (!aligned(qkv, 16) || !aligned(out, nq_bits ? 16 : 8))
        return fail(ARCQ_ERR_ALIGN, "%s: qkv must be 16-byte, out %d-byte aligned", fn, nq_bits ? 16 : 8);
    if (B > 65535 || H > (1 << 20) || B * n * 3 * H * head_dim >= (int64_t(1) << 40))
        return fail(ARCQ_ERR_SHAPE, "%s: tensor too large", fn);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int b = static_cast<int>(B), nn = static_cast<int>(n), hh = static_cast<int>(H);
    if (fp8) {
        if (nq_bits == 4) launch_attention_n<4, true>(qkv, out, b, nn, hh, scale, thr, cb, st);
        else if (nq_bits == 3) launch_attention_n<3, true>(qkv, out, b, nn, hh, scale, thr, cb, st);
        else launch_attention_n<2, true>(qkv, out, b, nn, hh, scale, thr, cb, st);
    } else if (nq_bits == 0) launch_attention_n<0>(qkv, out, b, nn, hh, scale, thr, cb, st);
    else if (nq_bits == 4) launch_attention_n<4>(qkv, out, b, nn, hh, scale, thr, cb, st);
    else if (nq_bits == 3) launch_attention_n<3>(qkv, out, b, nn, hh, scale, thr, cb, st);
    else launch_attention_n<2>(qkv, out, b, nn, hh, scale, thr, cb, st);
    return launch_status(fn);
}

}  // namespace
}  // namespace arcq

using namespace arcq;

ARCQ_API int arcq_attention_fwd(const void *qkv, void *out, int64_t B, int64_t n, int64_t H, int64_t head_dim, float scale,
                                void *stream)
{
    return attention_checked("arcq_attention_fwd", qkv, out, B, n, H, head_dim, scale, 0, nullptr, nullptr, stream);
}

ARCQ_API int arcq_attention_quant_fwd(const void *qkv, const float *thresholds, const float *codebook, int bits, void *x_hat,
                                      int64_t B, int64_t n, int64_t H, int64_t head_dim, float scale, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_attention_quant_fwd: bits must be 2, 3, or 4");
    if (B * n >= (int64_t(1) << 26)) return fail(ARCQ_ERR_SHAPE, "arcq_attention_quant_fwd: tensor too large");
    return attention_checked("arcq_attention_quant_fwd", qkv, x_hat, B, n, H, head_dim, scale, bits, thresholds, codebook, stream);
}

ARCQ_API int arcq_attention_quant_fp8_fwd(const void *qkv, const float *thresholds, const float *codebook, int bits, void *x8,
                                          int64_t B, int64_t n, int64_t H, int64_t head_dim, float scale, void *stream)
{
    if (!bits_ok(bits)) return fail(ARCQ_ERR_BITS, "arcq_attention_quant_fp8_fwd: bits must be 2, 3, or 4");
    if (B * n >= (int64_t(1) << 26)) return fail(ARCQ_ERR_SHAPE, "arcq_attention_quant_fp8_fwd: tensor too large");
    return attention_checked("arcq_attention_quant_fp8_fwd", qkv, x8, B, n, H, head_dim, scale, bits, thresholds, codebook, stream, true);
}
