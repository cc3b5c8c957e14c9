// What the kernels share in which a workgroup owns 64 rows and the launch's workgroups rebuild the weights between them: the
// pieces of w_hat, the counters by which a workgroup learns that all pieces are written, and how many workgroups a device holds.
#pragma once

#include "arcq_common.h"

#include <mutex>
#include <vector>

namespace arcq {

constexpr unsigned long long kEpoch = 1ull << 20;     // what one launch adds to its counter, whatever its grid

// One layer's packed weights and where their reconstruction goes.
struct WeightShare {
    const uint8_t *pw;                  // packed codes [N, K*bits/8]
    const float *cb, *wc, *ws, *wcs;
    __half *out;                        // block layout
};

// Piece idx of the block-layout w_hat, idx = ((n / 32) * (K / 8) + k / 8) * 32 + n % 32, holds w_hat[n][k .. k + 8):
// value (cb[code] - code_sum/64) * scale + center with one fma (FQ/arcq_packed_triton.py:59-74), stored at
// out + 8 idx, written through to memory.  In two steps so that the loads of the first can travel under other work.
struct Piece {
    uint32_t w;
    float c, s, m;
};
template <int BITS, int G>
__device__ __forceinline__ void fetch_piece(const WeightShare &p, int64_t idx, Piece &pc)
{
    constexpr int K = 64 * G, P = K / 8, pcols = K * BITS / 8;     // compile-time: the divisions below are multiplications
    const uint32_t i = static_cast<uint32_t>(idx);                 // N * K / 8 < 2^23 (N <= 16384, K <= 3072)
    const uint32_t r = i & 31u;
    const uint32_t t = i >> 5;
    const uint32_t nb = t / P;
    const uint32_t pp = t - nb * P;
    const uint32_t n = nb * 32u + r;
    pc.w = load_codes8<BITS>(p.pw + n * pcols + pp * BITS);
    const uint32_t mi = n * G + (pp >> 3);
    pc.c = p.wc[mi];
    pc.s = p.ws[mi];
    pc.m = p.wcs[mi] * 0.015625f;      // code_sum / 64, exact
}
template <int BITS>
__device__ __forceinline__ void finish_piece(const WeightShare &p, int64_t idx, const Piece &pc)
{
    constexpr int L = 1 << BITS;
    float cbv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) cbv[q] = p.cb[(pc.w >> (BITS * q)) & (L - 1)];      // 64 bytes, cached
    uint32_t out[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const __half2 h = __floats2half2_rn(fma_f32(cbv[2 * q] - pc.m, pc.s, pc.c), fma_f32(cbv[2 * q + 1] - pc.m, pc.s, pc.c));
        out[q] = *reinterpret_cast<const uint32_t *>(&h);
    }
    store_writethrough16(p.out + idx * 8, out[0], out[1], out[2], out[3]);
}

// Two counter words (zero when the code object is loaded) that belong to weight workspace `key` on the current device, nullptr if none
// is left, and the device's count of workgroups whose wait ran out.
unsigned long long *rows_counters_for(const void *key, unsigned long long **timeouts);

// Workgroups of `Kernel` (threads, dynamic LDS bytes) the current device holds at once.  A launch must not be larger:
// every workgroup waits for the weight shares of all the others, and those that are not resident write theirs only
// after a resident one has given up waiting (correct, but milliseconds late).  Asked once per device, kernel and LDS
// size; 0 if the runtime cannot tell.
template <auto Kernel>
inline int resident_workgroups(int threads, size_t smem)
{
    struct Entry { int dev; size_t smem; int blocks; };
    static std::mutex mutex;
    static std::vector<Entry> known;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(mutex);
    for (const Entry &e : known)
        if (e.dev == dev && e.smem == smem) return e.blocks;
    int per_cu = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void *>(Kernel), threads, smem) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        per_cu = cus = 0;
    known.push_back({dev, smem, per_cu * cus});
    return per_cu * cus;
}

}  // namespace arcq
