// Stage-1 arithmetic shared by the stand-alone activation quantizer and the fused small-M layer kernel
// (semantics: EXT/arcq_activation_kernel.cu:24-184): per-workgroup lookup tables and the per-group routine
// that turns 64 inputs held in one lane's registers into mu, s, the codes and the reconstructed values.
#pragma once

#include "arcq_common.h"

#include <type_traits>

namespace arcq {

// ---- FP8 operands (OCP E4M3) ---------------------------------------------------------------------------------------
constexpr float kFp8Max = 448.0f;

// Eight floats -> eight FP8 (E4M3, round to nearest even, finite values saturating at +-448, NaN kept) in two dwords.
__device__ __forceinline__ void to_fp8x8(const float (&v)[8], uint32_t &lo, uint32_t &hi)
{
    float c[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = v[i] != v[i] ? v[i] : fminf(fmaxf(v[i], -kFp8Max), kFp8Max);      // (NaN stays NaN)
    int a = 0, b = 0;
    a = __builtin_amdgcn_cvt_pk_fp8_f32(c[0], c[1], a, false);
    a = __builtin_amdgcn_cvt_pk_fp8_f32(c[2], c[3], a, true);
    b = __builtin_amdgcn_cvt_pk_fp8_f32(c[4], c[5], b, false);
    b = __builtin_amdgcn_cvt_pk_fp8_f32(c[6], c[7], b, true);
    lo = static_cast<uint32_t>(a);
    hi = static_cast<uint32_t>(b);
}

// Sixteen reconstructed values s (v[j0 + e] - code_mean) + mu as one 16-byte piece.
template <int N>
__device__ __forceinline__ void xhat_fp8x16(const float (&v)[N], int j0, float s, float code_mean, float mu, uint32_t (&o)[4])
{
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float t[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) t[e] = fma_f32(s, v[j0 + 8 * p + e] - code_mean, mu);
        to_fp8x8(t, o[2 * p], o[2 * p + 1]);
    }
}

// Values rounded to fp16 and widened again, two to a conversion.
template <int N>
__device__ __forceinline__ void round_to_half(float (&v)[N])
{
#pragma unroll
    for (int j = 0; j < N; j += 2) {
        const __half2 h = __floats2half2_rn(v[j], v[j + 1]);
        v[j] = __low2float(h), v[j + 1] = __high2float(h);
    }
}

constexpr int kMaxBuckets = 512;   // table entries 0 .. nb (nb <= 512); entry nb is reached by t == 8 only

// Bucket geometry: t in [-8, 8] maps to floor(f), f = t * scale + 8 * scale rounded to a multiple of 1/8; nb = 16 * scale
// buckets can hold a threshold.  The scale is the smallest of 4, 8, 16, 32 buckets per unit of t that separates every
// pair of thresholds (scale * smallest gap > 1), so the usual codebooks need a 65- or 129-entry table instead of 513.
// f is formed as 2^20 + f in one fma: in that binade a float's unit in the last place is 1/8, so the low mantissa bits
// of the result ARE 8 * f -- the byte offset of an 8-byte table entry once the three fraction bits are masked off.
// The map t -> bucket is monotone (fma and the mask are).  t = d/s itself is not formed: f comes from d and an approximate 1/s, which
// puts a value into its bucket or, within 2^-15 of an edge, into the one beside it; no threshold lies as close to an edge, so both
// give the same code.
constexpr float kBucketBias = 1048576.0f;      // 2^20
constexpr float kEdgeMargin = 0x1p-12f;        // between a threshold and the edges of its bucket, in buckets
struct BucketScale { float scale, offset; int nb; };      // offset = 8 * scale + 2^20, or 1/4 more (exact)

__device__ __forceinline__ BucketScale bucket_scale_for(float gap)      // gap: the smallest between neighbouring thresholds
{
    float scale = 32.0f;
    if (gap * 16.0f > 1.0f) scale = 16.0f;
    if (gap * 8.0f > 1.0f) scale = 8.0f;
    if (gap * 4.0f > 1.0f) scale = 4.0f;
    BucketScale q;
    q.scale = scale;
    q.offset = 8.0f * scale + kBucketBias;
    q.nb = static_cast<int>(16.0f * scale);
    return q;
}

// Bucket of a threshold: any float; -1 / nb flag a threshold outside [-8, 8).
__device__ __forceinline__ int bucket_of_threshold(float t, const BucketScale &q)
{
    const float f = __fmaf_rn(t, q.scale, q.offset);
    if (!(f >= kBucketBias)) return -1;         // below the table, or NaN
    if (f >= kBucketBias + static_cast<float>(q.nb)) return q.nb;
    return __float2int_rz(f - kBucketBias);     // exact difference
}

// Whether a threshold lies next to an edge (f rounds to a multiple of 1/8: the edges are at b - 1/16).
__device__ __forceinline__ bool near_an_edge(float t, const BucketScale &q)
{
    const float f = __fmaf_rn(t, q.scale, (q.offset - kBucketBias) - 8.0f * q.scale + 0.0625f);
    return !(fabsf(f - rintf(f)) >= kEdgeMargin);
}

// `u`: the threshold inside the bucket (+inf if none), or for a negative one the next float above it; `base`: 4 times the number of
// thresholds in lower buckets.
struct alignas(8) Bucket { float u; int base; };

// RN(d / s) > T, the quotient rounded to nearest, without a division: it holds exactly where d / s lies beyond T + h, h half the
// distance from T to the next float above (a quotient is never halfway between two floats), that is where s u - d + s e 2^-24 < 0
// with u = T, e = 2^k in T's binade for T >= 0, and u the next float, e = -2^k for T < 0: in both cases e is u without its mantissa.
// The first difference is a remainder, exact where it is small enough to matter, so the sign of the second is right: with
// 2^-60 <= s <= 2^58, T = 0 or |T| >= 2^-60, d = 0 or |d| >= 2^-90.  (A quotient rounded to nearest takes a product and four fused
// corrections where this takes two and a mask: 10 instructions a value with the lookup, now 7.  Stage 1 with a LayerNorm
// 12 608 x 768 16.1 -> 15.3 us, 50 432 x 1 024 58.0 -> 55.5; behind a product with GELU, 50 432 x 1 024 -> 4 096 616 -> 596 us.)
struct CodeScale { float s, s24, to_bucket; };
__device__ __forceinline__ CodeScale code_scale_of(float s, float about_1_over_s, const BucketScale &q)
{
    return CodeScale{s, s * 0x1p-24f, about_1_over_s * q.scale};
}
// The bucket of d.  In range |d / s| <= 8, f lies in [0, nb] <= 512.25 and the bucket's offset is bits 3..12 of the biased sum.
__device__ __forceinline__ Bucket bucket_of(float d, const CodeScale &c, const BucketScale &q, const Bucket *table)
{
    static_assert(sizeof(Bucket) == 8, "the offset assumes 8-byte table entries");
    const uint32_t at = __float_as_uint(__fmaf_rn(d, c.to_bucket, q.offset)) & 0x1ff8u;
    return *reinterpret_cast<const Bucket *>(reinterpret_cast<const char *>(table) + at);
}
// 4 times the code of d, whose bucket is bk.
__device__ __forceinline__ uint32_t code_offset_in(const Bucket &bk, float d, const CodeScale &c)
{
    const float e = __uint_as_float(__float_as_uint(bk.u) & 0xff800000u);
    const float r = __fmaf_rn(c.s24, e, __fmaf_rn(c.s, bk.u, -d));
    uint32_t below = __float_as_uint(r) >> 31;
    asm("" : "+v"(below));      // (a shift and one v_lshl_add; left alone the two shifts become one shift, a mask and an addition)
    return (below << 2) + static_cast<uint32_t>(bk.base);
}
__device__ __forceinline__ uint32_t code_offset_of(float d, const CodeScale &c, const BucketScale &q, const Bucket *table)
{
    return code_offset_in(bucket_of(d, c, q, table), d, c);
}
__device__ __forceinline__ float code_value(const float *cb, uint32_t offset)
{
    return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(cb) + offset);
}

// A quantizer's lookup tables in LDS.  `cb` needs no copy per lane: a read of 16 different entries meets no bank twice.
template <int ENTRIES>
struct QuantTablesOf {
    float cb[16], thr[16];      // (thr: the thresholds, or their running maxima where the buckets are not usable)
    BucketScale geometry;
    int usable;                      // 0: two thresholds in one bucket, one outside [-8, 8) or at an edge or tiny, or unsorted ones
    uint32_t holds[18];              // bit b: bucket b holds a threshold
    Bucket bucket[ENTRIES];
};
using QuantTables = QuantTablesOf<kMaxBuckets + 1>;

// A lane's threshold and codebook value, requested ahead of everything else that the building wave loads (loads complete in the
// order of their issue: behind a tile's, the tables of a launch of 12 608 x 1 536 values are 0.6 us late).
struct QuantParams { float thr, cb; };
template <int BITS>
__device__ __forceinline__ QuantParams load_quant_params(const float *__restrict__ thr, const float *__restrict__ cb, int lane)
{
    constexpr int L = 1 << BITS;
    return QuantParams{lane < L - 1 ? thr[lane] : __builtin_huge_valf(), lane < L ? cb[lane] : 0.0f};
}

// Table construction by ONE complete wave; the caller synchronizes.  Lane i takes threshold i: the smallest gap and the order come
// from its neighbour's lane, a bit per occupied bucket meets in LDS, and a bucket's number of lower thresholds is the count of
// lower bits (v_mbcnt).  (Every thread of up to four waves used to go over all thresholds, 15 uniform branches and 95 instructions
// per 64 buckets with a scalar hazard wait in each: 1.0 us of the 7.8 us that 197 x 384 values with a LayerNorm take.)
template <int BITS, int ENTRIES>
__device__ __forceinline__ void build_quant_tables(const QuantParams &p, QuantTablesOf<ENTRIES> &q, int lane)
{
    constexpr int L = 1 << BITS;
    constexpr float inf = __builtin_huge_valf();
    const float t = p.thr;
    if (lane < 18) q.holds[lane] = 0;
    auto dpp = [](float old, float v, auto ctrl) __attribute__((always_inline)) {
        return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, false));
    };
    const float next = dpp(inf, t, std::integral_constant<int, 0x101>{});        // row_shl:1, lane i + 1's
    const bool pair = lane < L - 2;
    bool bad = pair && !(t <= next);
    float gap = fminf(pair ? next - t : 16.0f, 16.0f);                           // (NaN gaps are ignored: `bad` has them)
    gap = fminf(gap, dpp(gap, gap, std::integral_constant<int, 0x121>{}));       // row_ror: the minimum of the sixteen lanes
    gap = fminf(gap, dpp(gap, gap, std::integral_constant<int, 0x122>{}));
    gap = fminf(gap, dpp(gap, gap, std::integral_constant<int, 0x124>{}));
    gap = fminf(gap, dpp(gap, gap, std::integral_constant<int, 0x128>{}));
    BucketScale g = bucket_scale_for(__int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(gap))));
    if (__any(lane < L - 1 && near_an_edge(t, g))) g.offset += 0.25f;
    const int tb = bucket_of_threshold(t, g);
    const bool inside = tb >= 0 && tb < g.nb;
    __builtin_amdgcn_wave_barrier();
    if (lane < L - 1) {
        bad = bad || !inside || near_an_edge(t, g) || (t != 0.0f && fabsf(t) < 0x1p-60f);
        const uint32_t bit = 1u << (tb & 31);
        if (inside) bad = bad || (atomicOr(&q.holds[tb >> 5], bit) & bit);
    }
    const bool usable = !__any(bad);
    float thr_or_max = t;
    if (!usable) {                                                               // the running maximum (infinite from a NaN on)
        if (t != t) thr_or_max = inf;
        thr_or_max = fmaxf(thr_or_max, dpp(-inf, thr_or_max, std::integral_constant<int, 0x111>{}));      // row_shr
        thr_or_max = fmaxf(thr_or_max, dpp(-inf, thr_or_max, std::integral_constant<int, 0x112>{}));
        thr_or_max = fmaxf(thr_or_max, dpp(-inf, thr_or_max, std::integral_constant<int, 0x114>{}));
        thr_or_max = fmaxf(thr_or_max, dpp(-inf, thr_or_max, std::integral_constant<int, 0x118>{}));
    }
    if (lane < 16) q.thr[lane] = thr_or_max, q.cb[lane] = p.cb;
    if (lane == 0) q.geometry = g, q.usable = usable;
    __builtin_amdgcn_wave_barrier();
    int below = 0;                                                               // thresholds in the buckets before b0
    for (int b0 = 0; b0 <= g.nb; b0 += 64) {
        const uint32_t lo = q.holds[b0 >> 5], hi = q.holds[(b0 >> 5) + 1];
        const int base = static_cast<int>(__builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, below)));
        const float thr = (((lane < 32 ? lo : hi) >> (lane & 31)) & 1u) ? q.thr[min(base, 15)] : inf;
        Bucket e;
        e.u = thr < 0.0f ? __int_as_float(__float_as_int(thr) - 1) : thr + 0.0f;      // (-0 as 0)
        e.base = 4 * base;
        if (b0 + lane <= g.nb) q.bucket[b0 + lane] = e;
        below += __popc(lo) + __popc(hi);
    }
}

// One group per lane, first half: xv holds the 64 inputs on entry and the residuals d_j = x_j - mu on exit.
// Needs no table, so it can run while other waves are still building them.
__device__ __forceinline__ void group_stats64(float (&xv)[64], float eps, float &mu_out, float &var_out, float &s_out)
{
    float mu = 0.0f;
#pragma unroll
    for (int j = 0; j < 64; ++j) mu += xv[j];
    mu *= 0.015625f;                       // exact: /64
    float var = 0.0f;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
        xv[j] -= mu;                       // d_j
        var += xv[j] * xv[j];
    }
    mu_out = mu;
    var_out = var;
    s_out = sqrtf(var * 0.015625f + eps);
}

// Codes without the buckets, for thresholds that these cannot hold: while (c < L - 1 && t > thr[c]) ++c stops at the first threshold
// that is not below t, so c counts the thresholds whose running maximum is.  The maxima ascend (q.thr holds them then, infinities from
// a NaN on): a bisection, one lookup, a comparison and two more instructions for each bit of the code.  (Every threshold in turn:
// packed codes of 50 432 x 1 024 fp32 at four bits 96 us at a comparison and an addition each, 57 now, 40 with usable buckets; behind a
// product with GELU, 6 304 x 1 024 -> 4 096, 101 us, 88 with usable buckets.)  Returns 4 times the codes.
template <int BITS, int N>
__device__ __forceinline__ void bisect_codes(const float (&t)[N], const float *maxima, uint32_t (&at)[N])
{
    constexpr uint32_t top = 4u << (BITS - 1);
    const float middle = maxima[(1 << (BITS - 1)) - 1];
#pragma unroll
    for (int e = 0; e < N; ++e) at[e] = t[e] > middle ? top : 0u;
#pragma unroll
    for (uint32_t step = top / 2; step >= 4; step /= 2) {
        float m[N];
#pragma unroll
        for (int e = 0; e < N; ++e) m[e] = code_value(maxima + step / 4 - 1, at[e]);
#pragma unroll
        for (int e = 0; e < N; ++e) at[e] += t[e] > m[e] ? step : 0u;
    }
}
// xv holds the residuals on entry and cb[code_j] on exit; put(j, code).  BATCH values at a time (registers).
template <int BITS, int BATCH = 8, int N, typename Put>
__device__ __forceinline__ void search_codes(float (&xv)[N], float s, const QuantTables &q, const Put &put)
{
    constexpr int B = N < BATCH ? N : BATCH;
#pragma unroll
    for (int j0 = 0; j0 < N; j0 += B) {
        float t[B];
        uint32_t at[B];
#pragma unroll
        for (int e = 0; e < B; ++e) t[e] = xv[j0 + e] / s;
        bisect_codes<BITS>(t, q.thr, at);
#pragma unroll
        for (int e = 0; e < B; ++e) {
            xv[j0 + e] = code_value(q.cb, at[e]);
            put(j0 + e, at[e] >> 2);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// The lookups of 64 values for a wave that has its SIMD for itself (or shares it with one that multiplies): the first read of eight
// values, the second read of the eight before and the sum of the eight before those are under way at a time, so that no read is waited
// for.  xv as in group_codes64; returns the sum.  A wave's 64 x 64 values beside another one's product: 9 300 -> 8 700 clocks.
__device__ __forceinline__ float codes64_in_turns(float (&xv)[64], const CodeScale &cs, const QuantTables &q, const BucketScale &bq)
{
    float sum = 0.0f;
    Bucket bk[2][8];
#pragma unroll
    for (int b = 0; b < 10; ++b) {
        if (b < 8) {
#pragma unroll
            for (int e = 0; e < 8; ++e) bk[b & 1][e] = bucket_of(xv[8 * b + e], cs, bq, q.bucket);
        }
        if (b >= 2) {
#pragma unroll
            for (int e = 0; e < 8; ++e) sum += xv[8 * (b - 2) + e];
        }
        __builtin_amdgcn_sched_barrier(0);
        if (b >= 1 && b < 9) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                float &v = xv[8 * (b - 1) + e];
                v = code_value(q.cb, code_offset_in(bk[(b - 1) & 1][e], v, cs));
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    return sum;
}

// Second half: xv holds the residuals on entry and cb[code_j] on exit.  The whole wave must call it (the fast/slow
// decision is wave-uniform).  `bq`, `table_ok`: q.geometry and q.usable, in registers.  BATCH: how many lookups may be in flight
// (all of them take registers that a product's accumulators leave no room for).  `code`: the codes, a byte each.
// BATCH = 0: codes64_in_turns.
template <int BITS, bool CODES, int BATCH = 64>
__device__ __forceinline__ void group_codes64(float (&xv)[64], float mu, float var, float s, const QuantTables &q, const BucketScale &bq,
                                              bool table_ok, float &sum_out, uint32_t (&code)[CODES ? 16 : 1])
{
    // The range that code_offset_of asks for: |d_j| >= 2^-90 whenever |mu| >= 2^-66, or all d_j are zero.
    const bool lane_fast = (s >= 0x1p-60f) && (s <= 0x1p58f) && !(fabsf(mu) < 0x1p-66f && var > 0.0f);
    const bool fast = table_ok && __all(lane_fast);
    auto put = [&](int j, uint32_t c) __attribute__((always_inline)) { code[j / 4] = j % 4 == 0 ? c : code[j / 4] | c << (8 * (j % 4)); };

    float sum_codes = 0.0f;
    if (fast) {
        const CodeScale cs = code_scale_of(s, __builtin_amdgcn_rcpf(s), bq);
        if constexpr (BATCH == 0) {
            static_assert(!CODES, "codes64_in_turns keeps none");
            sum_codes = codes64_in_turns(xv, cs, q, bq);
        } else {
#pragma unroll
            for (int j = 0; j < 64; ++j) {
                const uint32_t c = code_offset_of(xv[j], cs, bq, q.bucket);
                if constexpr (CODES) put(j, c >> 2);
                const float v = code_value(q.cb, c);
                xv[j] = v;
                sum_codes += v;
                if (BATCH < 64 && j % BATCH == BATCH - 1) __builtin_amdgcn_sched_barrier(0);
            }
        }
    } else {
        search_codes<BITS>(xv, s, q, [&](int j, uint32_t c) __attribute__((always_inline)) {
            if constexpr (CODES) put(j, c);
            sum_codes += xv[j];
        });
    }
    sum_out = sum_codes;
}

// ---- two lanes per group -------------------------------------------------------------------------------------
// For launches too small to fill the chip the length of one lane's instruction chain is what counts.  Lanes 2i and
// 2i + 1 then share group i: the even lane holds inputs 0..31, the odd lane inputs 32..63.  The per-element work
// halves; the three group sums keep their serial left-to-right order by running in two phases (the even lane folds
// its half from 0, hands the partial sum to the odd lane, which folds its half on top; every lane executes both
// phases and the phase that is not its own is discarded), so every result bit is the one-lane routine's.
__device__ __forceinline__ float from_even_lane(float v)     // the pair's even lane's value, in both lanes
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xA0, 0xf, 0xf, false));    // quad_perm [0,0,2,2]
}
__device__ __forceinline__ float from_odd_lane(float v)      // the pair's odd lane's value, in both lanes
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xF5, 0xf, 0xf, false));    // quad_perm [1,1,3,3]
}

// Serial sum of the group's 64 values v_0 + v_1 + ... (from 0.0f, left to right), this lane holding its half.
__device__ __forceinline__ float pair_serial_sum(const float (&v)[32])
{
    float a = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) a += v[j];           // even lane: values 0..31
    float b = from_even_lane(a);
#pragma unroll
    for (int j = 0; j < 32; ++j) b += v[j];           // odd lane: ... + values 32..63
    return from_odd_lane(b);
}

// xv: this lane's 32 inputs on entry, the residuals d_j = x_j - mu on exit; mu, var, s as group_stats64, in both lanes.
__device__ __forceinline__ void group_stats32x2(float (&xv)[32], float eps, float &mu_out, float &var_out, float &s_out)
{
    const float mu = pair_serial_sum(xv) * 0.015625f;     // exact: /64
    float sq[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        xv[j] -= mu;
        sq[j] = xv[j] * xv[j];
    }
    const float var = pair_serial_sum(sq);
    mu_out = mu;
    var_out = var;
    s_out = sqrtf(var * 0.015625f + eps);
}

// xv: residuals on entry, cb[code_j] on exit; sum_out = the serial sum of all 64 cb[code_j], in both lanes.  The
// whole wave must call it (the fast/slow decision is wave-uniform).  CODE_BITS != 0: the 32 codes too, packed CODE_BITS apart
// into `words`.
template <int BITS, int CODE_BITS = 0, int BATCH = 8>
__device__ __forceinline__ void group_codes32x2(float (&xv)[32], float mu, float var, float s, const QuantTables &q, const BucketScale &bq,
                                                bool table_ok, float &sum_out, uint32_t *words = nullptr)
{
    auto put = [&](int j, uint32_t c) __attribute__((always_inline)) {
        if constexpr (CODE_BITS != 0) {
            const int bit = j * CODE_BITS, d = bit >> 5, sh = bit & 31;
            words[d] = sh == 0 ? c : words[d] | (c << sh);
            if (sh + CODE_BITS > 32) words[d + 1] = c >> (32 - sh);
        }
    };
    const bool lane_fast = (s >= 0x1p-60f) && (s <= 0x1p58f) && !(fabsf(mu) < 0x1p-66f && var > 0.0f);      // (as above)
    const bool fast = table_ok && __all(lane_fast);
    if (fast) {
        const CodeScale cs = code_scale_of(s, __builtin_amdgcn_rcpf(s), bq);
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const uint32_t c = code_offset_of(xv[j], cs, bq, q.bucket);
            xv[j] = code_value(q.cb, c);
            put(j, c >> 2);
        }
    } else {
        search_codes<BITS, BATCH>(xv, s, q, put);
    }
    sum_out = pair_serial_sum(xv);
}

// ---- four, eight or sixteen lanes per group -------------------------------------------------------------------------------
// Where a launch leaves most of the chip idle: the serial sums stay as long (in LANES phases, a lane's partial sum handed to its
// neighbour after each; what a lane adds in a phase that is not its own is discarded), everything else of a value is spread.
// 197 x 384 values with a LayerNorm in front: 6.3 us with two lanes a group, 4.3 with eight.
template <int CTRL> __device__ __forceinline__ float lane_moved(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// v_0 + v_1 + ... over LANES neighbouring lanes (aligned), from 0.0f, left to right: valid in the last of them.
template <int LANES, int V>
__device__ __forceinline__ float lanes_serial_sum(const float (&v)[V])
{
    float a = 0.0f;
#pragma unroll
    for (int p = 0; p < LANES; ++p) {
        if (p > 0) a = lane_moved<0x111>(a);                   // row_shr:1
#pragma unroll
        for (int j = 0; j < V; ++j) a += v[j];
    }
    return a;
}
template <int LANES>
__device__ __forceinline__ float from_last_lane(float v, int lane)
{
    static_assert(LANES == 2 || LANES == 4 || LANES == 8 || LANES == 16, "lanes per group");
    if constexpr (LANES == 2) return from_odd_lane(v);
    if constexpr (LANES == 16) return lane_moved<0x15F>(v);    // row_newbcast:15
    const float quad = lane_moved<0xFF>(v);                    // quad_perm [3,3,3,3]
    if constexpr (LANES == 4) return quad;
    const float other = lane_moved<0x141>(quad);               // row_half_mirror (not inside the choice: every lane has to take part)
    return (lane & 4) ? quad : other;
}
template <int LANES>
__device__ __forceinline__ void group_stats_lanes(float (&xv)[64 / LANES], float eps, int lane, float &mu_out, float &var_out, float &s_out)
{
    constexpr int V = 64 / LANES;
    const float mu = from_last_lane<LANES>(lanes_serial_sum<LANES>(xv), lane) * 0.015625f;
    float sq[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        xv[j] -= mu;
        sq[j] = xv[j] * xv[j];
    }
    const float var = from_last_lane<LANES>(lanes_serial_sum<LANES>(sq), lane);
    mu_out = mu;
    var_out = var;
    s_out = sqrtf(var * 0.015625f + eps);
}
template <int BITS, int LANES>
__device__ __forceinline__ void group_codes_lanes(float (&xv)[64 / LANES], float mu, float var, float s, const QuantTables &q,
                                                  const BucketScale &bq, bool table_ok, int lane, float &sum_out)
{
    constexpr int V = 64 / LANES;
    const bool lane_fast = (s >= 0x1p-60f) && (s <= 0x1p58f) && !(fabsf(mu) < 0x1p-66f && var > 0.0f);      // (as above)
    if (table_ok && __all(lane_fast)) {
        const CodeScale cs = code_scale_of(s, __builtin_amdgcn_rcpf(s), bq);
#pragma unroll
        for (int j = 0; j < V; ++j) xv[j] = code_value(q.cb, code_offset_of(xv[j], cs, bq, q.bucket));
    } else {
        search_codes<BITS>(xv, s, q, [](int, uint32_t) __attribute__((always_inline)) {});
    }
    sum_out = from_last_lane<LANES>(lanes_serial_sum<LANES>(xv), lane);
}

// ---- stage 1 of the NEXT layer inside a GEMM's epilogue ----------------------------------------------------------
// The block-layout GEMM kernels stage their outputs 32 rows x 64 fp16 columns at a time in a wave-private LDS tile
// (`pitch` bytes per row) -- one quantization group per row.  When the layer's output is only ever consumed quantized
// (fc1 -> GELU -> fc2) the wave quantizes the staged chunk right there, exactly as the consuming layer's stage 1 would
// have done on the stored tensor (two lanes per group, same arithmetic, same bits), and writes x_hat into the
// consumer's 32-row block layout.  The consumer's lookup tables live in LDS (built once per workgroup by
// next_quant_setup).
// LDS of the consumer's quantizer.
constexpr int next_quant_lds_bytes() { return (static_cast<int>(sizeof(QuantTables)) + 15) / 16 * 16; }

// One wave of the workgroup makes the consumer's lookup tables in `lds` (next_quant_lds_bytes() bytes, 16-byte aligned), before a
// barrier that precedes the first epilogue.
template <int BITS>
__device__ __forceinline__ void next_quant_setup(const QuantParams &p, unsigned char *lds, int lane)
{
    build_quant_tables<BITS>(p, *reinterpret_cast<QuantTables *>(lds), lane);
}

// The consumer's stage 1 of a group that 64 / V neighbouring lanes (aligned) hold in registers, V fp16-rounded values each: v is
// replaced by the reconstruction.
template <int BITS, int V>
__device__ __forceinline__ void next_quant_lanes(const unsigned char *lds, float (&v)[V], int lane, float eps)
{
    constexpr int LANES = 64 / V;
    const QuantTables &q = *reinterpret_cast<const QuantTables *>(lds);
    float mu, var, s, sum;
    group_stats_lanes<LANES>(v, eps, lane, mu, var, s);
    group_codes_lanes<BITS, LANES>(v, mu, var, s, q, q.geometry, q.usable != 0, lane, sum);
    const float code_mean = sum * 0.015625f;
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = fma_f32(s, v[j] - code_mean, mu);
}

// One staged chunk (32 rows x 64 fp16 values, the rows `pitch` bytes apart) -> x_hat of the consuming layer.
// `gelu`: the exact GELU of the staged (rounded) values first, rounded to fp16 again.  dst = the chunk's first 16-byte
// piece of this lane's row (lane / 2) in the consumer's block layout, whose pieces are `rows` rows apart; `live` = whether
// the row is stored.  F8: the consumer's operands are FP8 (16 values a piece); `pad`: the chunk is the last of a row whose
// length is an odd number of groups, and the row's padding to 128 values is written too.  The whole wave calls it.
template <int BITS, bool F8 = false>
__device__ __forceinline__ void next_quant_rows(const unsigned char *lds, const unsigned char *stage, int pitch, int lane, bool gelu, float eps,
                                                void *dst, int rows, bool live, bool pad = false)
{
    typedef uint32_t u32x4_nq __attribute__((ext_vector_type(4)));
    const QuantTables &q = *reinterpret_cast<const QuantTables *>(lds);
    const BucketScale bq = q.geometry;
    const bool usable = q.usable != 0;
    const int r = lane >> 1, hf = lane & 1;
    float v[32];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const u32x4_nq w = *reinterpret_cast<const u32x4_nq *>(stage + r * pitch + hf * 64 + i * 16);
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            v[8 * i + 2 * d] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] & 0xffffu)));
            v[8 * i + 2 * d + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(w[d] >> 16)));
        }
    }
    if (gelu) {
#pragma unroll
        for (int i = 0; i < 4; ++i) gelu_of_halves(v + 8 * i);
        round_to_half(v);
    }
    float mu, var, s, sum;
    group_stats32x2(v, eps, mu, var, s);
    group_codes32x2<BITS>(v, mu, var, s, q, bq, usable, sum);
    const float code_mean = sum * 0.015625f;
    char *out = static_cast<char *>(dst);
    if constexpr (F8) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t o[4];
            xhat_fp8x16(v, 16 * i, s, code_mean, mu, o);
            if (live) store_writethrough16(out + static_cast<int64_t>(hf * 2 + i) * rows * 16, o[0], o[1], o[2], o[3]);
            if (live && pad) store_writethrough16(out + static_cast<int64_t>(4 + hf * 2 + i) * rows * 16, 0, 0, 0, 0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t o[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int j = 8 * i + 2 * d;
                const __half2 h = __floats2half2_rn(fma_f32(s, v[j] - code_mean, mu), fma_f32(s, v[j + 1] - code_mean, mu));
                o[d] = *reinterpret_cast<const uint32_t *>(&h);
            }
            if (live) store_writethrough16(out + static_cast<int64_t>(hf * 4 + i) * rows * 16, o[0], o[1], o[2], o[3]);
        }
    }
}

// The same for a chunk whose 32 rows are block `blk` of the consumer's operand at x_hat (N values a row, M rows): c0 = the
// chunk's first column.
template <int BITS, bool F8>
__device__ __forceinline__ void next_quant_block(const unsigned char *lds, const unsigned char *stage, int pitch,
                                                 int lane, bool gelu, float eps, void *x_hat, int blk, int M, int N, int c0)
{
    const int r = lane >> 1, rows = min(32, M - blk * 32);
    const int row_bytes = F8 ? (N + 127) / 128 * 128 : N * 2;
    char *dst = static_cast<char *>(x_hat) + static_cast<int64_t>(blk) * 32 * row_bytes + (static_cast<int64_t>(F8 ? c0 / 16 : c0 / 8) * rows + r) * 16;
    next_quant_rows<BITS, F8>(lds, stage, pitch, lane, gelu, eps, dst, rows, r < rows, F8 && c0 + 64 == N && (N & 64) != 0);
}

// ---- the same with a lane per group: two staged chunks at once ----
// Two lanes a group run each of the three serial sums twice (3 instructions a value).  Where a wave has two chunks of the same 32
// rows, lane l takes row l % 32 of chunk l / 32 instead: half a wave fetches its rows while the chunk is staged, the arithmetic runs
// once for both.  12 608 x 384 -> 1 536 with GELU 38.3 -> 35.3 us, 3 152 x 768 -> 3 072 38.3 -> 34.3, 6 304 x 1 024 -> 4 096
// 85.7 -> 83.0.
struct StagedGroup { uint32_t w[32]; };      // 64 fp16 values
__device__ __forceinline__ void take_staged_group(StagedGroup &g, const unsigned char *stage, int pitch, int lane, int chunk)
{
    typedef uint32_t u32x4_nq __attribute__((ext_vector_type(4)));
    if ((lane >> 5) == chunk) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u32x4_nq w = *reinterpret_cast<const u32x4_nq *>(stage + (lane & 31) * pitch + i * 16);
#pragma unroll
            for (int d = 0; d < 4; ++d) g.w[4 * i + d] = w[d];
        }
    }
}
// c0 = the first chunk's first column.  The whole wave calls it.
template <int BITS, bool F8>
__device__ __forceinline__ void next_quant_groups(const unsigned char *lds, const StagedGroup &g, int lane, bool gelu, float eps, void *x_hat,
                                                  int blk, int M, int N, int c0)
{
    const QuantTables &q = *reinterpret_cast<const QuantTables *>(lds);
    const BucketScale bq = q.geometry;
    const bool usable = q.usable != 0;
    float v[64];
#pragma unroll
    for (int d = 0; d < 32; ++d) {
        v[2 * d] = __half2float(__ushort_as_half(static_cast<unsigned short>(g.w[d] & 0xffffu)));
        v[2 * d + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(g.w[d] >> 16)));
    }
    if (gelu) {
#pragma unroll
        for (int i = 0; i < 8; ++i) gelu_of_halves(v + 8 * i);
        round_to_half(v);
    }
    float mu, var, s, sum;
    uint32_t none[1];
    group_stats64(v, eps, mu, var, s);
    group_codes64<BITS, false, 16>(v, mu, var, s, q, bq, usable, sum, none);
    const float code_mean = sum * 0.015625f;
    const int r = lane & 31, rows = min(32, M - blk * 32), c = c0 + 64 * (lane >> 5);
    const bool live = r < rows && c < N;
    const int row_bytes = F8 ? (N + 127) / 128 * 128 : N * 2;
    char *dst = static_cast<char *>(x_hat) + static_cast<int64_t>(blk) * 32 * row_bytes + (static_cast<int64_t>(F8 ? c / 16 : c / 8) * rows + r) * 16;
    if (!live) return;
    if constexpr (F8) {
        const bool pad = c + 64 == N && (N & 64) != 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t o[4];
            xhat_fp8x16(v, 16 * i, s, code_mean, mu, o);
            store_writethrough16(dst + static_cast<int64_t>(i) * rows * 16, o[0], o[1], o[2], o[3]);
            if (pad) store_writethrough16(dst + static_cast<int64_t>(4 + i) * rows * 16, 0, 0, 0, 0);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t o[4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const int j = 8 * i + 2 * d;
                const __half2 h = __floats2half2_rn(fma_f32(s, v[j] - code_mean, mu), fma_f32(s, v[j + 1] - code_mean, mu));
                o[d] = *reinterpret_cast<const uint32_t *>(&h);
            }
            store_writethrough16(dst + static_cast<int64_t>(i) * rows * 16, o[0], o[1], o[2], o[3]);
        }
    }
}

// ---- a row per lane, straight from a wave's 64 x 64 tile of a product ----
// A 2 x 2 tile of 32 x 32 MFMA blocks (acc[column block][row block], operand roles swapped: lane (l % 32, l / 32) holds row l % 32 of a
// row block at columns 8 t + 4 (l / 32) + c) is one quantization group of 64 rows.  One v_permlane32_swap per pair of values gives lane
// l all of row l: no trip through LDS, and the quantizer's serial sums run once.
typedef float mfma_block_t __attribute__((ext_vector_type(16)));
// SCALED: products are multiplied by `scale` first.  bias: of the tile's first column.  row: fp16 pairs.
template <bool SCALED>
__device__ __forceinline__ void tile_to_rows(const mfma_block_t (&acc)[2][2], float scale, const float *bias, int lane, uint32_t (&row)[32])
{
    const int lh = lane >> 5;
    uint32_t w[2][2][8];                     // [row block, later the half][column block][pair of columns]
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const float4 b = *reinterpret_cast<const float4 *>(bias + cb * 32 + 8 * t + 4 * lh);
            const float b4[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const float lo = acc[cb][rb][4 * t + 2 * d], hi = acc[cb][rb][4 * t + 2 * d + 1];
                    const __half2 h = SCALED ? __floats2half2_rn(lo * scale + b4[2 * d], hi * scale + b4[2 * d + 1])
                                             : __floats2half2_rn(lo + b4[2 * d], hi + b4[2 * d + 1]);
                    w[rb][cb][2 * t + d] = *reinterpret_cast<const uint32_t *>(&h);
                }
        }
#pragma unroll
    for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // The lower lanes keep row block 0 and take its other columns, the upper ones row block 1.
            const auto r = __builtin_amdgcn_permlane32_swap(w[0][cb][i], w[1][cb][i], false, false);
            const int pair = cb * 16 + 4 * (i >> 1) + (i & 1);
            row[pair] = r[0], row[pair + 2] = r[1];
        }
}
__device__ __forceinline__ void widen(const uint32_t *pairs, float *v, int n)
{
#pragma unroll
    for (int i = 0; i < n; ++i) {
        v[2 * i] = __half2float(__ushort_as_half(static_cast<unsigned short>(pairs[i] & 0xffffu)));
        v[2 * i + 1] = __half2float(__ushort_as_half(static_cast<unsigned short>(pairs[i] >> 16)));
    }
}
__device__ __forceinline__ uint32_t half_pair(float a, float b)
{
    const __half2 h = __floats2half2_rn(a, b);
    return *reinterpret_cast<const uint32_t *>(&h);
}
// GELU of the row's values 8 FROM .. 8 TO.
template <int FROM, int TO>
__device__ __forceinline__ void gelu_pairs(uint32_t (&row)[32])
{
#pragma unroll
    for (int o = FROM; o < TO; ++o) {
        float v[8];
        widen(row + 4 * o, v, 4);
        gelu_of_halves(v);
#pragma unroll
        for (int i = 0; i < 4; ++i) row[4 * o + i] = half_pair(v[2 * i], v[2 * i + 1]);
        __builtin_amdgcn_sched_barrier(0);
    }
}
// Stage 1 of the row's group: x_hat as fp16 pairs, or (F8) as FP8.  The whole wave calls it.
template <int BITS, bool F8>
__device__ __forceinline__ void quantize_row(const uint32_t (&row)[32], const QuantTables &q, float eps, uint32_t (&out)[F8 ? 16 : 32])
{
    float v[64];
    widen(row, v, 32);
    float mu, var, s, sum;
    uint32_t none[1];
    const BucketScale geometry = q.geometry;
    const bool usable = q.usable != 0;
    group_stats64(v, eps, mu, var, s);
    group_codes64<BITS, false, 0>(v, mu, var, s, q, geometry, usable, sum, none);
    const float code_mean = sum * 0.015625f;
    if constexpr (F8) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t o[4];
            xhat_fp8x16(v, 16 * i, s, code_mean, mu, o);
#pragma unroll
            for (int e = 0; e < 4; ++e) out[4 * i + e] = o[e];
        }
    } else {
#pragma unroll
        for (int i = 0; i < 32; ++i) out[i] = half_pair(fma_f32(s, v[2 * i] - code_mean, mu), fma_f32(s, v[2 * i + 1] - code_mean, mu));
    }
}

}  // namespace arcq
