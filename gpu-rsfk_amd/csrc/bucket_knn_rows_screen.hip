// Bucket K-NN for buckets whose points fit into LDS whole, trees after the first ones of a build: the pairs are bounded on the
// matrix cores first.  Same function and same results as bucket_knn_rows.hip (which has the first trees, and any call on rows that
// are not sorted yet); K <= 64, rows sorted.
//
// In a later tree few candidates of a bucket can still enter a row (10M x 32, K = 32, buckets of 64..256, 10 trees: one in eight
// in the third tree, one in thirty in the last), and the kernel that runs the fp32 chain of every candidate from both ends was
// bound by the vector instructions of those chains and of one-by-one insertions (89 % busy).  Here:
//
//   1. the fp32 rows of the bucket are staged into LDS (pitch an odd number of 16-byte units).
//   2. A wavefront takes 32 members at a time against all tiles of 32 candidates.  The rows minus a common point (the mean of 16 of
//      them), times a power of two s that puts the longest of them between 2^13 and 2^14, are rounded to float16 on the fly;
//      v_mfma_f32_32x32x16_f16 accumulates the products.  With x = s (a - m), y = s (b - m), S = |x|^2 + |y|^2, R the longest and G the
//      accumulated product of the rounded vectors,
//          | s^2 |a - b|^2 - (S - 2 G) |  <=  c S + z,
//          c = 1.05 * 2^-10 + (4 D16 + 16) 2^-23,  z = 4.1 h sqrt(D) R + 2.1 h^2 D,  h = 2^-14     (D16 = D rounded up to 16):
//      two roundings of at most 2^-11 per product give (2^-10 + 2^-22) S, the differences 2^-23 S, accumulation and norms at most
//      1.7 (D16 + 2) 2^-23 S; z is for values below the least normal number h, wherever they end up.  The fp32 chain returns at least
//      (1 - gamma) times the real-number distance, gamma = (D + 8) 2^-22.
//      The pair is dropped iff ((1 - c) S - 2 G) > s^2 last slot / (1 - gamma) + z; for a lane that is one comparison per pair: the
//      accumulator starts at -(1 - c)|y|^2 / 2 and is compared with ((1 - c)|x|^2 - s^2 last slot / (1 - gamma) - z) / 2.  A norm of
//      1e37 or more, or NaN, drops nothing.  A lane holds the outcome for one member (a column of the tile) as bits.
//      (bfloat16 needs no s, but its c is eight times as large and leaves more pairs to the exact chains: 10M x 32, trees 3 to 10 31.6 -> 30.5 ms.)
//   3. The bits become a list of pairs ordered by member.  A turn takes up to 64 of them, whole members, one pair per lane: the exact
//      chains from LDS, the members' K-NN rows (up to 256 slots) to LDS, then every lane counts the entries of its row below its
//      candidate (one 64-bit comparison of (distance, index) each), sees whether the row holds the candidate already, and counts the member's
//      other new candidates below it.  That is the candidate's slot; an entry of the row moves up by the candidates that end below it.
//      Nothing is inserted one by one: walking the candidates of one member after the other, with the row in registers, took 12.1 ms
//      for the third tree and 4.1 for the last where this takes 7.8 and 2.8 (470 and 125 scalar instructions per row, now 80 and 28).
//   4. The slots of changed rows are stored in full lines.
//
// One workgroup per bucket, no barrier after the norms; a row is owned by one wavefront.  LDS for three workgroups per compute unit
// (42 pieces of 1,280 bytes at D = 32: 128 bytes more mean two workgroups, and the last tree takes 4.1 ms instead of 2.8).
//
// 10M x 32, K = 32, buckets of 64..256, 10 trees, trees 3 to 10: 10.0 8.6 7.8 7.4 7.1 6.8 6.6 6.4 -> 7.4 4.9 3.9 3.4 3.1 2.9 2.8 2.7 ms;
// loading and storing every row of a tree's buckets alone takes 2.1 ms, the rest is vector instructions (93 per row in the last tree, 244 in the
// third; 400 and 600 before).  Requesting the rows of the next turn during this one: 12 % slower.
#include "rsfk_common.hpp"
#include "knn_list.hpp"
#include "mfma_split.hpp"
#include "forest.hpp"
#include "bucket_knn_stage.hpp"
#include "bucket_knn_turn.hpp"
#include <algorithm>
#include <cmath>

namespace rsfk {

namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kListCap = 256;                 // pairs on a wavefront's list: at least the candidates of one member

// Per wavefront.
template <int KS>
struct WaveLds : TurnLds {
    uint16_t list[kListCap];                  // pairs: member << 8 | candidate
    float mean[16 * KS];                      // the common point
};

// NT: buckets of up to 64 NT points; KS: steps of 16 dimensions.
template <int NT, int KS>
__global__ __launch_bounds__(kRowsThreads, 3) void k_bucket_knn_rows_screen(const float* __restrict__ points, int D, int K,
                                                                             const int* __restrict__ ids, const int* __restrict__ starts,
                                                                             const int* __restrict__ sizes, int min_size, int max_size,
                                                                             int* __restrict__ knn_idx, float* __restrict__ knn_dist,
                                                                             int pitch, int per_k, uint32_t per_np, float c_err, float over, float lost)
{
    extern __shared__ __align__(16) float lds_r[];
    float* rows = lds_r;                                          // 64 NT rows of `pitch` floats
    int* lids = reinterpret_cast<int*>(lds_r + 64 * NT * pitch);
    float* nhalf = reinterpret_cast<float*>(lids + 64 * NT);      // -(1 - c)|y|^2 / 2 per point
    WaveLds<KS>& L = reinterpret_cast<WaveLds<KS>*>(nhalf + 64 * NT)[threadIdx.x >> 6];

    const int s = sizes[blockIdx.x];
    if (s < min_size || s > max_size || s < 2) return;
    const int* bid = ids + (size_t)starts[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 31, half = lane >> 5;
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);
    const int np = (D + 3) >> 2;                                  // 16-byte pieces per row

    for (int i = tid; i < 64 * NT; i += kRowsThreads) lids[i] = i < s ? bid[i] : -1;
    __syncthreads();
    // The last slots of this wavefront's members (lanes 0..31) and, so that the rows wait nearer when they are merged into, a
    // word of their indices (lanes 32..63): requested before anything else.
    float tau_of[NT > 2 ? 2 : 1];
#pragma unroll
    for (int t = 0; t < (NT > 2 ? 2 : 1); ++t) {
        const int m = 32 * (wave + kRowsWaves * t) + col;
        tau_of[t] = INFINITY;
        if (m < s) {
            const size_t at = (size_t)lids[m] * (size_t)K;
            tau_of[t] = half ? __int_as_float(knn_idx[at]) : knn_dist[at + (K - 1)];
        }
    }
    // (rows beyond s stay as they are: their pairs are masked out)
    stage_rows<kRowsThreads>(rows, pitch, lids, s, points, D, per_np, vec_ok);
    __syncthreads();

    // the common point: every wavefront works it out for itself, with the same result
#pragma unroll
    for (int c0 = 0; c0 < 16 * KS; c0 += 32) {
        const int c = c0 + col;
        float sum = 0.0f;
        if (c < 4 * np) {
#pragma unroll
            for (int k = 0; k < 8; ++k) sum += rows[(((2 * k + half) * s) >> 4) * pitch + c];
        }
        sum += __shfl_xor(sum, 32, 64);
        if (half == 0 && c < 16 * KS) L.mean[c] = sum * 0.0625f;          // (zero beyond the last dimension)
    }
    wave_lds_sync();
    // dimensions 16 k + 8 half .. of point r, minus the common point (times scale, once the mean is), and as operand of the matrix cores
    float scale = 1.0f;
    auto centred = [&](int r, int k, float (&x)[8]) {
        const float* p = rows + r * pitch + 16 * k + 8 * half;
        float4 a = *reinterpret_cast<const float4*>(p);
        float4 b = *reinterpret_cast<const float4*>(p + 4);
        if (k == KS - 1 || k >= 3) {                              // (five steps: 49 dimensions or more)
            const int left = np - 4 * k - 2 * half;               // pieces of the row from here on
            if (left < 1) a = make_float4(0.f, 0.f, 0.f, 0.f);
            if (left < 2) b = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const float4 ma = *reinterpret_cast<const float4*>(&L.mean[16 * k + 8 * half]);
        const float4 mb = *reinterpret_cast<const float4*>(&L.mean[16 * k + 8 * half + 4]);
        // (a power of two: s a - s m rounds as a - m does)
        x[0] = __builtin_fmaf(a.x, scale, -ma.x); x[1] = __builtin_fmaf(a.y, scale, -ma.y);
        x[2] = __builtin_fmaf(a.z, scale, -ma.z); x[3] = __builtin_fmaf(a.w, scale, -ma.w);
        x[4] = __builtin_fmaf(b.x, scale, -mb.x); x[5] = __builtin_fmaf(b.y, scale, -mb.y);
        x[6] = __builtin_fmaf(b.z, scale, -mb.z); x[7] = __builtin_fmaf(b.w, scale, -mb.w);
    };
    auto operand = [&](int r, int k) {
        float x[8];
        centred(r, k, x);
        typedef __attribute__((ext_vector_type(8))) float f32x8;
        const f32x8 v = {x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
        return __builtin_convertvector(v, f16x8);
    };
    for (int T = wave; 32 * T < s; T += kRowsWaves) {
        float n = 0.0f;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            float x[8];
            centred(32 * T + col, k, x);
#pragma unroll
            for (int u = 0; u < 8; ++u) n = __builtin_fmaf(x[u], x[u], n);
        }
        n += __shfl_xor(n, 32, 64);
        if (half == 0) nhalf[32 * T + col] = n;
    }
    __syncthreads();
    // s and R, the same for all wavefronts; from here on lengths are in units of s
    float far = 0.0f;
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const float n = 64 * u + lane < s ? nhalf[64 * u + lane] : 0.0f;
        far = n < 1e37f ? fmaxf(far, n) : far;
    }
    far = wave_max(far);
    const int e2 = (int)(__float_as_uint(far) >> 23) - 126;      // far < 2^e2
    scale = __uint_as_float((uint32_t)(127 + max(-60, min(60, 14 - ((e2 + 1) >> 1)))) << 23);
    const float scale2 = scale * scale;
    const float z = lost * (4.1f * scale * sqrtf(far) + 2.1f * lost);
    __syncthreads();                                              // the norms have been read
#pragma unroll
    for (int c0 = 0; c0 < 16 * KS; c0 += 64)
        if (c0 + lane < 16 * KS) L.mean[c0 + lane] *= scale;
    for (int T = wave; 32 * T < s; T += kRowsWaves)
        if (half == 0) {
            const float n = nhalf[32 * T + col];
            nhalf[32 * T + col] = n < 1e37f ? -0.5f * (1.0f - c_err) * n * scale2 : INFINITY;
        }
    __syncthreads();

    RowTurn turn(K, per_k);
    const int nj = (s + 31) >> 5;
    for (int T = wave; T < nj; T += kRowsWaves) {
        const int i = 32 * T + col;
        const int gid = lids[i];
        const float tau = __shfl(T < kRowsWaves ? tau_of[0] : tau_of[NT > 2 ? 1 : 0], col, 64);
        f16x8 mem[KS];
#pragma unroll
        for (int k = 0; k < KS; ++k) mem[k] = operand(i, k);
        const float limit = -nhalf[i] - 0.5f * ((tau * over + 1e-35f) * scale2 + z);
        uint32_t bits[NT];
#pragma unroll
        for (int w = 0; w < NT; ++w) {
            bits[w] = 0;
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int J = 2 * w + u;
                if (2 * w >= nj) break;                           // (both or none: their waits overlap)
                f32x16 g;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 v = *reinterpret_cast<const float4*>(nhalf + 32 * J + 8 * q + 4 * half);
                    g[4 * q] = v.x; g[4 * q + 1] = v.y; g[4 * q + 2] = v.z; g[4 * q + 3] = v.w;
                }
#pragma unroll
                for (int k = 0; k < KS; ++k)
                    g = __builtin_amdgcn_mfma_f32_32x32x16_f16(operand(32 * J + col, k), mem[k], g, 0, 0, 0);
                uint32_t b = 0;
#pragma unroll
                for (int r = 15; r >= 0; --r) b = b + b + (g[r] < limit ? 0u : 1u);
                // bit r: candidate 32 J + 8 (r / 4) + 4 half + r % 4
                if (J >= nj - 1) {
                    const int left = s - 32 * J - 4 * half;
                    uint32_t there = 0;
#pragma unroll
                    for (int q = 0; q < 4; ++q) there |= ((1u << min(4, max(0, left - 8 * q))) - 1u) << (4 * q);
                    b &= there;
                }
                if (J == T && half == ((col >> 2) & 1)) b &= ~(1u << (((col >> 3) << 2) + (col & 3)));
                bits[w] |= b << (16 * u);
            }
        }
        int mine = 0;
#pragma unroll
        for (int w = 0; w < NT; ++w) {
            if (i >= s) bits[w] = 0;
            mine += __popc(bits[w]);
        }
        const int both = mine + __shfl_xor(mine, 32, 64);         // candidates of this member
        const int upto = __shfl(wave_excl_scan_i(half == 0 ? both : 0), col, 64) + both;
        const int from = upto - both;                             // (both halves of the wavefront hold the members' numbers)
        const uint32_t act = (uint32_t)ballot64(both > 0);
        const int seq = __popc(act & ((1u << col) - 1u));         // members with candidates before this one

        for (int g0 = 0; g0 < 32;) {
            // members g0 .. g1 - 1: their pairs fit into the list (those of one always do)
            const int base = read_lane_i(from, g0);
            const int g1 = g0 + __popc((uint32_t)ballot64(upto - base <= kListCap) & (~0u << g0));
            wave_lds_sync();
            {
                int at = from - base + (half ? both - mine : 0);
                const bool in = col >= g0 && col < g1;
#pragma unroll
                for (int w = 0; w < NT; ++w) {
                    uint32_t b = in ? bits[w] : 0;
                    while (ballot64(b != 0) != 0) {
                        if (b != 0) {
                            const int r = __ffs(b) - 1;
                            b &= b - 1;
                            L.list[at++] = (uint16_t)((col << 8) | (64 * w + 4 * half + (r & 3) + ((r & 28) << 1)));
                        }
                    }
                }
            }
            for (int i0 = g0; i0 < g1;) {
                // members i0 .. i1 - 1: a lane per pair and room for the rows; or one member whose pairs take several turns
                const int first = read_lane_i(from, i0), seq0 = read_lane_i(seq, i0);
                const bool fits = upto - first <= 64 && seq + (both > 0 ? 1 : 0) - seq0 <= turn.n_room;
                const int i1 = i0 + max(1, __popc((uint32_t)ballot64(fits && col >= i0 && col < g1)));
                const int total = read_lane_i(upto, i1 - 1) - first;
                const bool act_here = both > 0 && col >= i0 && col < i1;
                const int n_rows = __popc((uint32_t)ballot64(act_here));
                i0 = i1;
                for (int e0 = 0; e0 < total; e0 += 64) {
                    const int n = min(64, total - e0);
                    wave_lds_sync();
                    if (act_here && half == 0) L.slot[seq - seq0] = make_int4(gid, 0, 0, 0);
                    wave_lds_sync();
                    turn.request(L, n_rows, knn_idx, knn_dist);
                    // the exact distances
                    const int entry = lane < n ? L.list[first - base + e0 + lane] : 0;
                    const int pcol = entry >> 8, j = entry & 255;
                    const int cid = lids[j];
                    float d = 0.0f;
                    {
                        const float* a = rows + (32 * T + pcol) * pitch;
                        const float* b = rows + j * pitch;
#pragma unroll 4
                        for (int q = 0; q < np; ++q) {
                            const float4 u = *reinterpret_cast<const float4*>(a + 4 * q), v = *reinterpret_cast<const float4*>(b + 4 * q);
                            float df;
                            df = u.x - v.x; d = __builtin_fmaf(df, df, d);
                            df = u.y - v.y; d = __builtin_fmaf(df, df, d);
                            df = u.z - v.z; d = __builtin_fmaf(df, df, d);
                            df = u.w - v.w; d = __builtin_fmaf(df, df, d);
                        }
                    }
                    const float last = __shfl(tau, pcol, 64);
                    const int lo = e0 > 0 ? 0 : __shfl(from, pcol, 64) - first;           // the member's pairs: lanes lo .. lo + count - 1
                    const int count = min(__shfl(both, pcol, 64), 64);
                    const int prow = __shfl(seq, pcol, 64) - seq0;
                    // (at the distance of the last slot the index decides: by the rank)
                    const bool enter = lane < n && d < INFINITY && d <= last;
                    turn.merge(L, n_rows, n, enter, prow, lo, count, cid, d, knn_idx, knn_dist);
                }
            }
            g0 = g1;
        }
    }
}

template <int NT, int KS>
int launch_cfg(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes, int n_buckets, int min_size,
               int max_size, int* knn_idx, float* knn_dist, hipStream_t stream)
{
    const int pitch = bucket_rows_pitch(D);
    const size_t lds = (size_t)64 * NT * (pitch + 2) * sizeof(float) + kRowsWaves * sizeof(WaveLds<KS>);
    const float c_err = 1.05f / 1024.0f + (float)(64 * KS + 16) / 8388608.0f;
    const float lost = std::sqrt((float)D) / 16384.0f;
    const double gamma = (double)(D + 8) / 4194304.0;
    const float over = (float)((1.0 + 1e-6) / (1.0 - gamma));
    auto kern = k_bucket_knn_rows_screen<NT, KS>;
    RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)n_buckets), dim3(kRowsThreads), lds, stream, points, D, K, ids, starts, sizes, min_size,
                       max_size, knn_idx, knn_dist, pitch, turn_per_k(K), rows_per_piece(D), c_err, over, lost);
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// Buckets of min_size..max_size points (others are skipped); max_size <= bucket_rows_cap(D, K).  Every K-NN row is sorted.
int launch_bucket_knn_rows_screen(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes,
                                  int n_buckets, int min_size, int max_size, int* knn_idx, float* knn_dist, hipStream_t stream)
{
    if (n_buckets <= 0 || max_size < 2) return 0;
    RSFK_CHECK(K >= 1 && K <= 64 && D >= 1, "bucket kernel with resident rows: K must be in 1..64 and D positive");
    RSFK_CHECK(max_size <= bucket_rows_cap(D, K), "bucket kernel with resident rows: buckets too large for the LDS");
    const int tiles = (max_size + 63) / 64;
#define RSFK_ROWS_CASE(NTV, KSV)                                                                                            \
    return launch_cfg<NTV, KSV>(points, D, K, ids, starts, sizes, n_buckets, min_size, max_size, knn_idx, knn_dist, stream)
    // (four tiles fit up to 36 dimensions, three up to 44, two up to 68)
    if (D <= 16) {
        if (tiles <= 2) RSFK_ROWS_CASE(2, 1);
        if (tiles == 3) RSFK_ROWS_CASE(3, 1);
        RSFK_ROWS_CASE(4, 1);
    }
    if (D <= 32) {
        if (tiles <= 2) RSFK_ROWS_CASE(2, 2);
        if (tiles == 3) RSFK_ROWS_CASE(3, 2);
        RSFK_ROWS_CASE(4, 2);
    }
    if (D <= 48) {
        if (tiles <= 2) RSFK_ROWS_CASE(2, 3);
        if (tiles == 3) RSFK_ROWS_CASE(3, 3);
        RSFK_ROWS_CASE(4, 3);
    }
    RSFK_CHECK(D <= 80 && tiles <= 2, "bucket kernel with resident rows: too many dimensions");
    RSFK_ROWS_CASE(2, 5);
#undef RSFK_ROWS_CASE
}

}  // namespace rsfk
