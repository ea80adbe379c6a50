// Bucket K-NN for buckets whose points fit into LDS whole (low-dimensional points,
// buckets of up to 256): same function and same results as the general kernel in
// bucket_knn.hip (see there for the reference kernels all of them replace), K <= 64.
//
// The tiled kernel looks at a bucket of s points as ceil(s / 64)^2 / 2 tiles of the
// pair matrix and visits the K-NN row of a point once per tile it takes part in:
// with buckets of 64..256 points a row is read, merged into and written about three
// times per tree, and with few trees over many points nearly every visit changes it.
// Here a row is touched once:
//
//   1. the fp32 rows of the whole bucket are staged into LDS (coalesced 16-byte
//      pieces; pitch an odd number of 16-byte units);
//   2. a wavefront takes two members at a time.  Lane l runs the sequential fused
//      multiply-add chains (arithmetic of euclidean_distance_sqr,
//      compute_knn_from_buckets.cu:40-54: a pair has the same distance value as in every
//      other kernel) of candidates l, 64 + l, ... against both members: the
//      candidate's values are read from LDS once for the two, the members' values are
//      the same in all lanes (broadcast reads).  Every pair is computed from both
//      ends, which at these dimensions costs less than carrying a distance matrix
//      through LDS and a second visit of the rows;
//   3. all candidates of a member are then offered to its row (knn_list.hpp), held
//      in registers, and the row is stored if it changed.  Where more than a few candidates are below
//      the row's last slot (the first trees of a build) the two are merged by counting (place_young).
//      The K-NN rows of the next two members are requested before the chains of these two start.
//
// No distance matrix, no flags, no barrier after the staging; a row is owned by
// one wavefront (no locks).
#include "rsfk_common.hpp"
#include "knn_list.hpp"
#include "forest.hpp"
#include "bucket_knn_stage.hpp"
#include <algorithm>

namespace rsfk {

namespace {

constexpr int kRowsThreads = 256;
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kRowsStep = 32;                 // dimensions of the two members held in registers at a time
constexpr int kRowsLdsBytes = 40 * 1024;      // four workgroups per compute unit

constexpr int kYoungLeast = 12;               // candidates below the last slot from which a row is merged by counting
// Rows that are not new: in few dimensions most points of the second tree's bucket that are near enough are in the row already, and the
// insertions drop those at little cost.  Calls of two trees of 1M points, buckets of 64..256, K = 32, before and with this: D = 2 3.82 and 3.65
// ms (4.9 by counting alone), 4 4.17 and 3.87, 6 4.36 and 4.02, 8 4.47 and 3.81, 32 4.86 and 4.08.
constexpr int kYoungDims = 6;

// NT = tiles of 64 candidates: buckets of up to 64 NT points.  Buckets outside min_size..max_size are left alone.
// DENSE: with the merge by counting (the first trees of a build; the code costs the later ones a few per cent when it is merely
// present).  Four wavefronts per SIMD: at three (130 registers) the first tree takes 11.7 ms, the second 13.0.
template <int NT, bool DENSE>
__global__ __launch_bounds__(kRowsThreads, 4) void k_bucket_knn_rows(const float* __restrict__ points, int D, int K,
                                                                   const int* __restrict__ ids, const int* __restrict__ starts,
                                                                   const int* __restrict__ sizes, int stride, int min_size,
                                                                   int max_size, int* __restrict__ knn_idx,
                                                                   float* __restrict__ knn_dist, int pitch, uint32_t per_np, int rows_sorted)
{
    extern __shared__ __align__(16) float lds_r[];
    float* rows = lds_r;                                          // 64 NT rows of `pitch` floats
    int* lids = reinterpret_cast<int*>(lds_r + 64 * NT * pitch);
    int* hist = lids + 64 * NT + 192 * (threadIdx.x >> 6);        // this wavefront's histogram, then 64 distances and 64 ids

    const int bkt = blockIdx.x;
    const int s = sizes[bkt];
    if (s < min_size || s > max_size || s < 2) return;
    const int* bid = ids + (starts ? (size_t)starts[bkt] : (size_t)bkt * (size_t)stride);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);
    const int np = (D + 3) >> 2;                                  // 16-byte pieces per row

    for (int i = tid; i < 64 * NT; i += kRowsThreads) lids[i] = i < s ? bid[i] : -1;
    __syncthreads();
    // rows beyond s stay as they are: their distances are never offered
    stage_rows<kRowsThreads>(rows, pitch, lids, s, points, D, per_np, vec_ok);
    __syncthreads();

    const int nt = (s + 63) >> 6;
    int cid[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) cid[t] = lids[64 * t + lane];

    // of member m: its id (the same in all lanes) and its row
    auto load_row = [&](int m, int& id, int& ri, float& rd) {
        id = __builtin_amdgcn_readfirstlane(lids[min(m, s - 1)]);
        ri = -2;
        rd = INFINITY;
        if (m < s && lane < K) {
            const size_t at = (size_t)id * (size_t)K + lane;
            ri = knn_idx[at];
            rd = knn_dist[at];
        }
    };
    // The row and its candidates by counting: false, with nothing done, where that does not pay or where more than 64 of them are
    // left.  A histogram over 64 equal intervals of the distances of the candidates below the last slot and of the row's entries
    // tells in which interval the K-th smallest lies; what is in later intervals has K others below it and cannot stay.  What is left
    // is put in the order of the intervals (a counting sort in LDS), and its place inside its interval found by looking at the
    // few others there.  Candidates that are points of the row already are found by a filter of 2,048 bits over the row's ids.
    // (10M x 32, buckets of 64..256: first tree 12.2 -> 10.6 ms, second, whose rows
    // used to take insertions, 14.1 -> 9.2; 530 and 470 vector instructions per point, 190 of them the chains.)
    auto place_young = [&](int id, const KnnRow<1>& row, bool (&ok)[NT], const float (&acc)[NT]) -> bool {
        bool in[NT];
        int n_in = 0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            // (no NaN and no infinite distance; one at the last slot may have the smaller index)
            in[t] = ok[t] && acc[t] <= row.tau && acc[t] < INFINITY;
            n_in += __popcll(ballot64(in[t]));
        }
        if (n_in < kYoungLeast || row.changed) return false;          // (a row that had to be put in order is stored whole)
        const bool mine = lane < K && row.idx[0] >= 0 && row.dist[0] < INFINITY;
        const int n_row = __popcll(ballot64(mine));
        // A row that holds nothing but, possibly, the point itself is new; any other entry may be a candidate too.  (Not told by the number
        // of entries: after a bucket of two points, or from the caller, a row's only entry is another point.)
        const bool new_row = ballot64(mine && row.idx[0] != id) == 0;
        const bool insert = !new_row && D < kYoungDims;              // the histogram of the candidates alone, then insertions
        if (insert && n_in <= K + 16) return false;
        if (ballot64(lane < K && row.idx[0] >= 0 && !mine) != 0) return false;
        // the intervals: from the least of them to the last slot of a full row, or to the mean of the candidates (to the largest, where
        // fewer than K are below the mean); what is beyond is in the last one
        float lo = !new_row && lane > 0 && mine ? row.dist[0] : INFINITY, sum = 0.0f;       // (not the point itself, which is at 0)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (in[t]) { lo = fminf(lo, acc[t]); sum += acc[t]; }
        lo = -wave_max(-lo);
        float hi = row.tau;
        if (row.tau_i < 0) {                                         // (an empty last slot, whatever distance stands there)
            hi = wave_total_f(sum) * __builtin_amdgcn_rcpf((float)n_in);
            int n_below = n_row;
#pragma unroll
            for (int t = 0; t < NT; ++t) n_below += __popcll(ballot64(in[t] && acc[t] < hi));
            if (n_below < K + 8) {
                hi = mine ? row.dist[0] : 0.0f;
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    if (in[t]) hi = fmaxf(hi, acc[t]);
                hi = wave_max(hi);
            }
        }
        if (!(hi > lo)) return false;
        const float scale = 63.5f / (hi - lo);
        auto bin_of = [&](float d) { return min(63, (int)(fmaxf(d - lo, 0.0f) * scale)); };   // does not decrease when the distance grows
        wave_lds_sync();
        hist[lane] = 0;
        wave_lds_sync();
        int bin[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            bin[t] = bin_of(acc[t]);
            if (in[t]) atomicAdd(&hist[bin[t]], 1);
        }
        const int bin_row = bin_of(row.dist[0]);
        if (mine && !insert) atomicAdd(&hist[bin_row], 1);
        wave_lds_sync();
        const int h = hist[lane];
        const int before = wave_excl_scan_i(h);
        const int all = n_in + n_row;
        const int need = insert ? K : min(all, K + (new_row ? 0 : 4));        // (some may be there twice)
        const int cross = first_lane(ballot64(before + h >= need));
        const int n_left = read_lane_i(before + h, cross);
        if (insert || n_left > 64) {
            // (insertions, of those that can stay)
            if (insert || new_row)
#pragma unroll
                for (int t = 0; t < NT; ++t) ok[t] = in[t] && bin[t] <= cross;
            return false;
        }
        wave_lds_sync();
        hist[lane] = before;
        wave_lds_sync();
        constexpr int kOfRow = (int)0x80000000;
        int2* left = reinterpret_cast<int2*>(hist + 64);              // (distance, id, with kOfRow for the row's own)
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (in[t] && bin[t] <= cross) left[atomicAdd(&hist[bin[t]], 1)] = make_int2(__float_as_int(acc[t]), cid[t]);
        if (mine && bin_row <= cross) left[atomicAdd(&hist[bin_row], 1)] = make_int2(__float_as_int(row.dist[0]), row.idx[0] | kOfRow);
        wave_lds_sync();
        const bool here = lane < n_left;
        const int2 v = here ? left[lane] : make_int2(0x7f800000, kOfRow);
        const float d = __int_as_float(v.x);
        const int c = v.y & ~kOfRow;
        const int b = here ? bin_of(d) : 0;
        int i = here && b > 0 ? hist[b - 1] : 0;                      // (hist: where the intervals end)
        const int end = here ? hist[b] : 0;
        int rank = i;
        while (ballot64(i < end) != 0) {
            if (i < end) {
                const int2 o = left[i];
                rank += pair_above(d, c, __int_as_float(o.x), o.y & ~kOfRow) ? 1 : 0;
                ++i;
            }
        }
        // candidates that are in the row: the filter first, then the row's ids
        bool twice = false;
        if (!new_row) {
            auto bit_of = [](int id) { return (id ^ (id >> 11)) & 2047; };
            wave_lds_sync();
            hist[lane] = 0;
            wave_lds_sync();
            if (mine) atomicOr(&hist[bit_of(row.idx[0]) >> 5], 1 << (bit_of(row.idx[0]) & 31));
            wave_lds_sync();
            uint64_t maybe = ballot64(v.y >= 0 && ((hist[bit_of(c) >> 5] >> (bit_of(c) & 31)) & 1));
            while (maybe) {
                const int j = first_lane(maybe);
                maybe &= maybe - 1;
                const int cj = read_lane_i(c, j);
                const bool held = ballot64(mine && row.idx[0] == cj) != 0;
                twice |= held && lane == j;
            }
        }
        uint64_t again = ballot64(twice);
        if (n_left < all && n_left - __popcll(again) < K) return false;       // (so many twice that the interval was too early)
        while (again) {
            const int j = first_lane(again);
            again &= again - 1;
            rank -= pair_above(d, c, read_lane_f(d, j), read_lane_i(c, j)) ? 1 : 0;
        }
        if (here && !twice && rank < K) {
            const size_t to = (size_t)id * (size_t)K + rank;
            knn_idx[to] = c;
            knn_dist[to] = d;
        }
        return true;
    };
    auto finish = [&](int m, int id, int ri, float rd, const float (&acc)[NT]) {
        KnnRow<1> row;
        row.idx[0] = ri;
        row.dist[0] = rd;
        if (rows_sorted) row.init_sorted(K);
        else row.init_from_regs(K);                               // rows that arrive unsorted are rebuilt here
        bool ok[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) ok[t] = t < nt && cid[t] >= 0 && 64 * t + lane != m;
        if (DENSE && place_young(id, row, ok, acc)) return;
        // tile after tile: the last slot a tile leaves behind already turns away candidates of the next
#pragma unroll
        for (int t = 0; t < NT; ++t)
            if (t < nt) row.merge(ok[t], cid[t], acc[t]);
        if (row.changed) {
            const size_t at = (size_t)id * (size_t)K;
            row.store(knn_idx + at, knn_dist + at);
        }
    };

    // members wave, wave + 4 (a pair), wave + 8, wave + 12 (the next pair), ...
    int id0, id1, nid0, nid1;
    int ri0, ri1, nri0, nri1;
    float rd0, rd1, nrd0, nrd1;
    load_row(wave, id0, ri0, rd0);
    load_row(wave + kRowsWaves, id1, ri1, rd1);
    for (int m0 = wave; m0 < s; m0 += 2 * kRowsWaves) {
        const int m1 = m0 + kRowsWaves;
        load_row(m0 + 2 * kRowsWaves, nid0, nri0, nrd0);
        load_row(m1 + 2 * kRowsWaves, nid1, nri1, nrd1);
        const bool two = m1 < s;
        const float* r0 = rows + m0 * pitch;
        const float* r1 = rows + (two ? m1 : m0) * pitch;
        float acc0[NT], acc1[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) { acc0[t] = 0.0f; acc1[t] = 0.0f; }
        for (int d0 = 0; d0 < 4 * np; d0 += kRowsStep) {
            const int nq = min(kRowsStep / 4, np - (d0 >> 2));
            float4 x0[kRowsStep / 4], x1[kRowsStep / 4];
#pragma unroll
            for (int q = 0; q < kRowsStep / 4; ++q) {
                if (q < nq) {
                    x0[q] = *reinterpret_cast<const float4*>(r0 + d0 + 4 * q);
                    x1[q] = *reinterpret_cast<const float4*>(r1 + d0 + 4 * q);
                }
            }
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (t < nt) {
                    const float* rc = rows + (64 * t + lane) * pitch + d0;
                    float a0 = acc0[t], a1 = acc1[t];
#pragma unroll
                    for (int q = 0; q < kRowsStep / 4; ++q) {
                        if (q < nq) {
                            const float4 v = *reinterpret_cast<const float4*>(rc + 4 * q);
                            float df;
                            df = x0[q].x - v.x; a0 = __builtin_fmaf(df, df, a0);
                            df = x0[q].y - v.y; a0 = __builtin_fmaf(df, df, a0);
                            df = x0[q].z - v.z; a0 = __builtin_fmaf(df, df, a0);
                            df = x0[q].w - v.w; a0 = __builtin_fmaf(df, df, a0);
                            df = x1[q].x - v.x; a1 = __builtin_fmaf(df, df, a1);
                            df = x1[q].y - v.y; a1 = __builtin_fmaf(df, df, a1);
                            df = x1[q].z - v.z; a1 = __builtin_fmaf(df, df, a1);
                            df = x1[q].w - v.w; a1 = __builtin_fmaf(df, df, a1);
                        }
                    }
                    acc0[t] = a0;
                    acc1[t] = a1;
                }
            }
        }
        finish(m0, id0, ri0, rd0, acc0);
        if (two) finish(m1, id1, ri1, rd1, acc1);
        id0 = nid0; ri0 = nri0; rd0 = nrd0;
        id1 = nid1; ri1 = nri1; rd1 = nrd1;
    }
}

template <int NT, bool DENSE>
int launch_rows_cfg(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes, int n_buckets,
                    int stride, int min_size, int max_size, int* knn_idx, float* knn_dist, int pitch, bool rows_sorted,
                    hipStream_t stream)
{
    const size_t lds = (size_t)64 * NT * pitch * sizeof(float) + (size_t)64 * (NT + 3 * kRowsWaves) * sizeof(int);
    auto kern = k_bucket_knn_rows<NT, DENSE>;
    RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3((unsigned)n_buckets), dim3(kRowsThreads), lds, stream, points, D, K, ids, starts, sizes, stride,
                       min_size, max_size, knn_idx, knn_dist, pitch, rows_per_piece(D), rows_sorted ? 1 : 0);
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// Floats from one staged row to the next.
int bucket_rows_pitch(int D)
{
    int pitch = (D + 3) & ~3;
    if (((pitch >> 2) & 1) == 0) pitch += 4;              // odd number of 16-byte units: rows start in different banks
    return pitch;
}

// Largest bucket the kernel takes for points of D dimensions and rows of K neighbours (0: none).
int bucket_rows_cap(int D, int K)
{
    if (K > 64) return 0;
    const int per_point = bucket_rows_pitch(D) * (int)sizeof(float) + (int)sizeof(int);
    const int tiles = std::min(4, (kRowsLdsBytes - 3 * 64 * kRowsWaves * (int)sizeof(int)) / (64 * per_point));
    return 64 * tiles;
}

// Buckets of min_size..max_size points (others are skipped); max_size <= bucket_rows_cap(D, K).  young_rows: the rows
// may be new or far from done (the first trees of a build, or unknown).
int launch_bucket_knn_rows(const float* points, int D, int K, const int* ids, const int* starts, const int* sizes, int n_buckets,
                           int stride, int min_size, int max_size, bool rows_sorted, bool young_rows, int* knn_idx,
                           float* knn_dist, hipStream_t stream)
{
    if (n_buckets <= 0 || max_size < 2) return 0;
    RSFK_CHECK(K >= 1 && K <= 64 && D >= 1, "bucket kernel with resident rows: K must be in 1..64 and D positive");
    RSFK_CHECK(max_size <= bucket_rows_cap(D, K), "bucket kernel with resident rows: buckets too large for the LDS");
    const int pitch = bucket_rows_pitch(D);
    const int tiles = (max_size + 63) / 64;
#define RSFK_ROWS_CASE(NTV, DV)                                                                                             \
    return launch_rows_cfg<NTV, DV>(points, D, K, ids, starts, sizes, n_buckets, stride, min_size, max_size, knn_idx, knn_dist, \
                                    pitch, rows_sorted, stream)
    if (young_rows) {
        if (tiles <= 2) RSFK_ROWS_CASE(2, true);
        if (tiles == 3) RSFK_ROWS_CASE(3, true);
        RSFK_ROWS_CASE(4, true);
    }
    if (tiles <= 2) RSFK_ROWS_CASE(2, false);
    if (tiles == 3) RSFK_ROWS_CASE(3, false);
    RSFK_ROWS_CASE(4, false);
#undef RSFK_ROWS_CASE
}

}  // namespace rsfk
