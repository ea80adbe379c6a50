// The fp32 rows of a bucket's s points (global indices in `lids`) to LDS, by a workgroup of THREADS threads: coalesced 16-byte pieces,
// rows of `pitch` floats, zeros up to the next multiple of four dimensions.  The pieces of four turns are requested together: with
// one at a time a bucket of 158 points x 32 waited five times for memory.
#pragma once
#include "rsfk_common.hpp"
#include "wave64.hpp"

namespace rsfk {

// 2^32 / (pieces of a row), rounded up: it / np = the upper half of it * per_np for the few thousand pieces of a bucket (D > 4; with one
// piece a row 0 stands for 2^32).
inline uint32_t rows_per_piece(int D)
{
    const uint64_t np = (uint64_t)(D + 3) >> 2;
    return (uint32_t)((((uint64_t)1 << 32) + np - 1) / np);
}

template <int THREADS>
__device__ __forceinline__ void stage_rows(float* rows, int pitch, const int* lids, int s, const float* __restrict__ points, int D,
                                           uint32_t per_np, bool vec_ok)
{
    constexpr int kAhead = 4;
    const int np = (D + 3) >> 2, n = s * np;
    for (int it0 = threadIdx.x; it0 < n; it0 += kAhead * THREADS) {
        float4 v[kAhead];
        int to[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int it = min(it0 + u * THREADS, n - 1);         // (the last piece again: the same value to the same place)
            const int m = per_np != 0 ? (int)__umulhi((uint32_t)it, per_np) : it, pc = it - m * np;
            to[u] = m * pitch + 4 * pc;
            v[u] = load_dims(points + (size_t)lids[m] * (size_t)D + 4 * pc, D - 4 * pc, vec_ok);
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) *reinterpret_cast<float4*>(&rows[to[u]]) = v[u];
    }
}

}  // namespace rsfk
