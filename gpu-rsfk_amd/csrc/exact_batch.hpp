// Exact distances of a batch of up to 64 candidates to one point, by one wavefront, and their merge into the
// point's K-NN row: shared by the exploration kernels and the query-set search.
//
// The candidates' fp32 rows are gathered with coalesced segments (several lanes per row), transposed through a
// tile in LDS, and every lane runs the sequential fused multiply-add chain of "its" candidate (the arithmetic
// of euclidean_distance_sqr, compute_knn_from_buckets.cu:40-54, so a pair of points has one distance value
// everywhere in the library).
#pragma once
#include "rsfk_common.hpp"
#include "knn_list.hpp"

namespace rsfk {

constexpr int kChunk = 32;              // fp32 dimensions per staging step (default)

struct ExploreLds {          // per wavefront; sizes fixed at launch
    int* table;              // hash set / candidate list, table_size ints
    int* srow;               // snapshot of the point's own row, K ints
    int* queue2;             // candidates that passed the screen, waiting for the exact distance
    float* xrow;             // the point's coordinates, zero padded to bf16_valid(D)
    float* tile;             // 64 x (chunk + 4) words
    double* rank;            // rank_words(SL) words for merge_ranked (exact_direct; exact_batch has them in its tile)
};

// Load one 16-byte piece (4 dimensions) of a candidate row, zero beyond D.
__device__ __forceinline__ float4 load_piece(const float* __restrict__ row, int d, int D, bool vec_ok)
{
    return d < D ? load_dims(row + d, D - d, vec_ok) : make_float4(0.f, 0.f, 0.f, 0.f);
}

// Exact distances of the first n candidates of `list` to the point, by one wavefront: lane l < ROWS has that of candidate l.  False: the
// sums were left where all of them were above limit.  CH = dimensions staged per step: a step moves ROWS rows x CH floats through the
// tile (ROWS (CH + 4) words).  DEEP: the loads of
// two steps are in flight while a third is being used (two register buffers that take turns, so that waiting for
// one does not wait for the other): for kernels with few wavefronts per SIMD, whose gathers would otherwise wait
// for each other.  GROUP: 16-byte pieces of a row whose reads from the tile are requested together (0: one at a time, the
// form that needs the fewest registers).
template <int CH, int ROWS, bool DEEP, int GROUP>
__device__ __forceinline__ bool exact_distances(float* tile, const float* xrow, const int* list, int n, const float* __restrict__ points,
                                                int D, bool vec_ok, float limit, float& acc)
{
    constexpr int kPieces = CH / 4;         // 16-byte pieces of a row per step = lanes per row
    constexpr int kRows = 64 / kPieces;     // rows per load instruction
    constexpr int kLoads = ROWS / kRows;    // load instructions per step
    constexpr int kP = CH + 4;              // tile pitch: odd number of 16-byte units
    const int lane = lane_id();
    const int sub = lane / kPieces;         // which of the rows of a load instruction
    const int piece = lane % kPieces;       // which 16-byte piece of the segment
    const float* rp[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int r = i * kRows + sub;
        rp[i] = r < n ? points + (size_t)list[r] * (size_t)D : nullptr;    // nothing is read for the rows beyond n
    }
    float4 pre[DEEP ? 2 : 1][kLoads];
    auto request = [&](float4 (&buf)[kLoads], int d0) {
        if (d0 < D) {
#pragma unroll
            for (int i = 0; i < kLoads; ++i)
                buf[i] = rp[i] ? load_piece(rp[i], d0 + piece * 4, D, vec_ok) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    acc = 0.0f;
    // one step: the buffer's values (dimensions d0 ..) go through the tile, the buffer is refilled with the step
    // `ahead` dimensions later, the chains advance.  Returns false when no candidate can enter any more.
    auto step = [&](float4 (&buf)[kLoads], int d0, int ahead) {
        wave_lds_sync();                 // previous step's tile reads are done
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            *reinterpret_cast<float4*>(&tile[(i * kRows + sub) * kP + piece * 4]) = buf[i];
        request(buf, d0 + ahead);
        wave_lds_sync();
        const int pieces = min(kPieces, (D - d0 + 3) >> 2);
        const float* mine = &tile[(ROWS < 64 ? lane & (ROWS - 1) : lane) * kP];
        const float* xs = &xrow[d0];
        auto chain4 = [&](const float4& a, const float4& x) {
            float df;
            df = a.x - x.x; acc = __builtin_fmaf(df, df, acc);
            df = a.y - x.y; acc = __builtin_fmaf(df, df, acc);
            df = a.z - x.z; acc = __builtin_fmaf(df, df, acc);
            df = a.w - x.w; acc = __builtin_fmaf(df, df, acc);
        };
        if (GROUP > 0 && pieces == kPieces) {
            // a whole step: the reads of the tile and of the point for 4 GROUP dimensions are requested together, so
            // that the chain waits for LDS once per group and not once per four dimensions (8 GROUP registers)
            constexpr int kGroup = GROUP > 0 ? GROUP : 1;
            static_assert(kPieces % kGroup == 0, "a step is a whole number of groups");
#pragma unroll
            for (int q0 = 0; q0 < kPieces; q0 += kGroup) {
                float4 a[kGroup], x[kGroup];
#pragma unroll
                for (int q = 0; q < kGroup; ++q) {
                    a[q] = *reinterpret_cast<const float4*>(mine + 4 * (q0 + q));
                    x[q] = *reinterpret_cast<const float4*>(xs + 4 * (q0 + q));
                }
#pragma unroll
                for (int q = 0; q < kGroup; ++q) chain4(a[q], x[q]);
            }
        } else {
            for (int q = 0; q < pieces; ++q)
                chain4(*reinterpret_cast<const float4*>(mine + 4 * q), *reinterpret_cast<const float4*>(xs + 4 * q));
        }
        // partial sums only grow: once all of them are above the limit nothing can enter
        return ballot64(lane < n && acc <= limit) != 0;
    };
    bool finished = true;
    request(pre[0], 0);
    if (DEEP) {
        request(pre[1], CH);
        for (int d0 = 0; d0 < D; d0 += 2 * CH) {
            if (!step(pre[0], d0, 2 * CH)) { finished = false; break; }
            if (d0 + CH < D && !step(pre[1], d0 + CH, 2 * CH)) { finished = false; break; }
        }
    } else {
        for (int d0 = 0; d0 < D; d0 += CH)
            if (!step(pre[0], d0, CH)) { finished = false; break; }
    }
    wave_lds_sync();
    return finished;
}

// The same for up to 64 candidates, which are then offered to the row.  tau_cap: a bound the caller
// knows for the row's final last slot (candidates above it need not be finished), else +inf.  RANK: no point of the list is in the row
// or on the list twice, but at this very distance: the batch is merged by merge_ranked.
template <int SL, int CH = kChunk, bool DEEP = false, int GROUP = 0, bool RANK = false>
__device__ __forceinline__ void exact_batch(const ExploreLds& L, const int* list, int n,
                                            const float* __restrict__ points, int D, bool vec_ok, KnnRow<SL>& row,
                                            float tau_cap = INFINITY)
{
    const int lane = lane_id();
    const int my_c = lane < n ? list[lane] : -1;
    float acc;
    // (unfinished sums are all above the last slot)
    const bool finished = exact_distances<CH, 64, DEEP, GROUP>(L.tile, L.xrow, list, n, points, D, vec_ok, fminf(row.tau, tau_cap), acc);
    if (RANK) {
        static_assert(!RANK || rank_words(SL) <= 64 * (CH + 4), "the ranks' working memory takes the place of the tile");
        row.merge_ranked(lane < n && finished, my_c, acc, reinterpret_cast<double*>(L.tile));
    } else {
        row.merge(lane < n && finished, my_c, acc);
    }
}

// Lanes with the bit give a and take b of the lane CTRL away, which gives b and takes a.
template <int CTRL>
__device__ __forceinline__ void quad_swap(float& a, float& b, bool bit)
{
    const float got = dpp_f<CTRL>(bit ? a : b);
    a = bit ? got : a;
    b = bit ? b : got;
}
template <int CTRL>
__device__ __forceinline__ void quad_swap(float4& a, float4& b, bool bit)
{
    quad_swap<CTRL>(a.x, b.x, bit);
    quad_swap<CTRL>(a.y, b.y, bit);
    quad_swap<CTRL>(a.z, b.z, bit);
    quad_swap<CTRL>(a.w, b.w, bit);
}

// The same without the tile: the chain of candidate l runs in the registers of lane l, 32 dimensions (eight 16-byte pieces) per step; the point's
// coordinates come from L.xrow (every lane reads the same word).  For short rows: no LDS besides xrow, no synchronisation inside the batch.
// QUADS: four lanes load 64 bytes of the row of each of them in turn and exchange the pieces; else a lane reads its own row, which the query-set search does
// where rows are short or few (ann.hip).  (A lane loading its own row asks for every line eight times, and
// a request of one lane takes the address units as long as one of four lanes in a row: they were busy 67 to 76 % of the exploration merge's time.  10M x 32
// 18.95 -> 17.33 ms, 1M x 100 2.56 -> 2.44, 1M x 256 5.95 -> 5.65, 123,457 x 37, K = 45 0.838 -> 0.660.  Whole lines by eight lanes each through 4 KB of LDS:
// 26.3, 3.57, 8.1, 1.11: 97 registers, and the LDS of four more wavefronts.)
template <int SL, bool QUADS, bool RANK = false>
__device__ __forceinline__ void exact_direct(const ExploreLds& L, const int* list, int n, const float* __restrict__ points,
                                             int D, bool vec_ok, KnnRow<SL>& row, float tau_cap = INFINITY)
{
    const int lane = lane_id();
    const int my_c = lane < n ? list[lane] : -1;
    const float* rp = points + (size_t)(my_c >= 0 ? my_c : 0) * (size_t)D;
    float acc = 0.0f;
    const float tau0 = fminf(row.tau, tau_cap);
    bool finished = true;
    // QUADS: instruction k of 16 dimensions loads 64 bytes of the row of lane k of every four lanes, and the four exchange them
    const int quarter = 4 * (lane & 3);
    const bool odd = (lane & 1) != 0, upper = (lane & 2) != 0;
    const int id[4] = {dpp_i<0x00>(my_c), dpp_i<0x55>(my_c), dpp_i<0xAA>(my_c), dpp_i<0xFF>(my_c)};
    // the four dimensions from d on, of this lane's candidate (xrow is zero beyond D like the pieces)
    const auto chain = [&](int d, const float4& v) {
        const float4 x = *reinterpret_cast<const float4*>(&L.xrow[d]);
        float df;
        df = v.x - x.x; acc = __builtin_fmaf(df, df, acc);
        df = v.y - x.y; acc = __builtin_fmaf(df, df, acc);
        df = v.z - x.z; acc = __builtin_fmaf(df, df, acc);
        df = v.w - x.w; acc = __builtin_fmaf(df, df, acc);
    };
    for (int d0 = 0; d0 < D; d0 += 32) {
        float4 v[8];
        if (!QUADS) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                v[i] = my_c >= 0 ? load_piece(rp, d0 + 4 * i, D, vec_ok) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (d0 + 4 * i < D) chain(d0 + 4 * i, v[i]);              // (wave-uniform)
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int d = d0 + 16 * (i >> 2) + quarter, k = id[i & 3];
                v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (k >= 0 && d < D) v[i] = load_dims(points + (size_t)(uint32_t)k * (size_t)(uint32_t)D + (size_t)(uint32_t)d, D - d, false);
            }
#pragma unroll
            for (int h = 0; h < 8; h += 4) {
                quad_swap<kDppXor1>(v[h], v[h + 1], odd);
                quad_swap<kDppXor1>(v[h + 2], v[h + 3], odd);
                quad_swap<kDppXor2>(v[h], v[h + 2], upper);
                quad_swap<kDppXor2>(v[h + 1], v[h + 3], upper);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = h; i < h + 4; ++i)
                    if (d0 + 4 * i < D) chain(d0 + 4 * i, v[i]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // partial sums only grow: once all of them are above the row maximum nothing can enter
        if (ballot64(lane < n && acc <= tau0) == 0) { finished = false; break; }
    }
    // (unfinished sums are all above the last slot)
    if (RANK) row.merge_ranked(lane < n && finished, my_c, acc, L.rank);
    else row.merge(lane < n && finished, my_c, acc);
}

}  // namespace rsfk
