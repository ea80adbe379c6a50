// Bucket K-NN of several trees at once, for inputs too small to fill the device with the buckets of one tree.
//
// The kernels that take a tree's buckets one tree after the other (bucket_knn_screen.hip and others) own a K-NN row
// inside a tree only, so the launches of a forest form a chain: at 3,000 x 200 a tree has 60 buckets for 256 compute
// units and every launch of the chain takes the 60 us one bucket takes (plus 27 us where two streams hand over to each
// other).  A row is the K smallest (distance, index) pairs of everything it is offered, in whatever order, so the
// chain is not needed:
//   k_forest_pairs   a workgroup per 64 x 64 tile of a bucket, all buckets of all trees of a group in one launch; the
//                    distances (every pair once, and its mirror image) go to memory, row j N + place of the member in
//                    the permutation of tree j, and info[p][j] says where the point p is in tree j;
//   k_forest_merge   a wavefront per point reads its rows of all trees, the loads of the next trees in flight, and
//                    merges them into the point's K-NN row, which is read and written once per group.
// A point meets a near neighbour in many trees: the ids a row has taken or turned away are kept in a small direct-mapped
// table in LDS, which drops the repeats of a whole tree with one read per lane (an id that was taken and fell out again
// is above the row's last pair for good, so a hit never has to be looked at again).  The first tree's candidates of a
// row that is new are placed by counting (small_bucket::place_by_rank) instead of being inserted one by one.
#include "rsfk_common.hpp"
#include "knn_list.hpp"
#include "forest.hpp"
#include "bucket_knn_tile.hpp"
#include "bucket_small_body.hpp"
#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace rsfk {

namespace {

struct alignas(16) PairsLds {
    union {
        struct {
            float a[kTile * kDCP];
            float b[kTile * kDCP];
        };
        float dist[kTile * kDistPitch];          // once the rows are no longer needed
    };
    int ida[kTile];
    int idb[kTile];
};

// stats: kTreeStatPitch ints per tree, {buckets of at most kBucketSplit points, larger ones, ...}: the former fill the front of the
// tree's leaf table, the latter its back.  tri: tiles on and above the diagonal of the largest bucket (of max_tiles by
// max_tiles tiles).
__global__ __launch_bounds__(256) void k_forest_pairs(const float* __restrict__ points, int N, int D, int T, const int* __restrict__ perm,
                                                       const int* __restrict__ leaf_start, const int* __restrict__ leaf_size,
                                                       int leaf_cap, const int* __restrict__ stats, int max_tiles, int tri,
                                                       int pitch, float* __restrict__ pair_dist, int2* __restrict__ info)
{
    __shared__ PairsLds L;
    const int j = blockIdx.y;
    const int n_small = stats[kTreeStatPitch * j], n_big = stats[kTreeStatPitch * j + 1];
    int slot = blockIdx.x, I = 0, J = 0;
    if (slot >= n_small) {
        const int y = slot - n_small, big = y / tri;
        if (big >= n_big) return;
        slot = leaf_cap - 1 - big;
        int t = y - big * tri;                    // tile (I, J) of place t in the order (0,0) (0,1) .. (0,T-1) (1,1) ..
        while (t >= max_tiles - I) { t -= max_tiles - I; ++I; }
        J = I + t;
    }
    const int start = leaf_start[(size_t)j * leaf_cap + slot], s = leaf_size[(size_t)j * leaf_cap + slot];
    if (J * kTile >= s) return;
    const int* bid = perm + (size_t)j * (size_t)N + start;
    const int tid = threadIdx.x;
    const int ty = tid >> 4, tx = tid & 15;
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);
    const int rows = min(kTile, s - I * kTile), cols = min(kTile, s - J * kTile);
    const bool diag = I == J;
    if (tid < kTile) {
        const int id = tid < rows ? bid[I * kTile + tid] : -1;
        L.ida[tid] = id;
        if (diag && id >= 0) info[(size_t)id * T + j] = make_int2(start, (I * kTile + tid) | (s << 16));
    } else if (tid < 2 * kTile) {
        L.idb[tid - kTile] = tid - kTile < cols ? bid[J * kTile + tid - kTile] : -1;
    }
    if (s < 2) return;
    float acc[4][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[r][c] = 0.0f;
    __syncthreads();
    pair_tile(L, points, D, rows, cols, diag, vec_ok, acc);
    // the tile -> LDS (the blocks below the diagonal of a diagonal tile are the mirror image of those above)
    const int nrb = (rows + 15) >> 4, ncb = (cols + 15) >> 4;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (r >= nrb || c >= ncb || (diag && c < r)) continue;
            const int i = ty + 16 * r, k = tx + 16 * c;
            L.dist[i * kDistPitch + k] = acc[r][c];
            if (diag && c > r) L.dist[k * kDistPitch + i] = acc[r][c];
        }
    __syncthreads();
    // ... -> the rows of the members of tile I, then, off the diagonal, of those of tile J
    float* M = pair_dist + ((size_t)j * (size_t)N + (size_t)start) * (size_t)pitch;
    const int lane = tid & 63, wave = tid >> 6;
    for (int i = wave; i < rows; i += 4)
        if (lane < cols) M[(size_t)(I * kTile + i) * pitch + J * kTile + lane] = L.dist[i * kDistPitch + lane];
    if (!diag)
        for (int i = wave; i < cols; i += 4)
            if (lane < rows) M[(size_t)(J * kTile + i) * pitch + I * kTile + lane] = L.dist[lane * kDistPitch + i];
}

constexpr int kSeen = 256;          // entries of a wavefront's table of ids that have been offered

__device__ __forceinline__ int seen_place(int id) { return (int)((uint32_t)id * 2654435761u >> 24); }

// A new row (nothing in it but, possibly, the point itself) from the distances of one bucket: dv[v] of lane l is the
// distance of candidate l + 64 v (the point itself included), +inf where there is none, n candidates, cv their ids.  When
// there are more than 64 SL of them, a distance is looked for by bisection that leaves at least K and at most 64 SL (a
// few steps: the window is wide); those are gathered in the lanes, ranked by counting and stored at their ranks.  False,
// with nothing changed, when no such distance was found or two distances are equal (insertions then).
// xi, xd: 64 SL words of LDS each.
template <int SL, int CL>
__device__ __forceinline__ bool new_row_by_rank(KnnRow<SL>& row, int K, const float (&dv)[CL], const int (&cv)[CL], int n, int* xi, float* xd,
                                                int* seen)
{
    const int lane = lane_id();
    constexpr int kCap = 64 * SL;
    float t = INFINITY;
    if (n > kCap) {
        float lo = INFINITY, hi = 0.0f;
#pragma unroll
        for (int v = 0; v < CL; ++v) {
            lo = fminf(lo, dv[v]);
            hi = fmaxf(hi, dv[v] < INFINITY ? dv[v] : 0.0f);
        }
        lo = -wave_max(-lo);
        hi = wave_max(hi);
        int count = 0;
        for (int it = 0; it < 12; ++it) {
            t = 0.5f * (lo + hi);
            count = 0;
#pragma unroll
            for (int v = 0; v < CL; ++v) count += __popcll(ballot64(dv[v] <= t));
            if (count > kCap) hi = t;
            else if (count < K) lo = t;
            else break;
        }
        if (count > kCap || count < K) return false;
    }
    int m = 0;
    wave_lds_sync();
#pragma unroll
    for (int v = 0; v < CL; ++v) {
        const bool take = dv[v] <= t && dv[v] < INFINITY;
        const uint64_t mask = ballot64(take);
        const int at = m + mask_prefix(mask);
        if (take) {
            xi[at] = cv[v];
            xd[at] = dv[v];
        }
        m += __popcll(mask);
    }
    wave_lds_sync();
    float cd[SL], place[SL];
    int ci[SL];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        const bool in = lane + 64 * s < m;
        cd[s] = in ? xd[lane + 64 * s] : INFINITY;
        ci[s] = in ? xi[lane + 64 * s] : -1;
        place[s] = cd[s];
    }
    if (!small_bucket::place_by_rank<SL>(place, m)) return false;
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        xi[lane + 64 * s] = lane + 64 * s < K ? -1 : -2;
        xd[lane + 64 * s] = INFINITY;
    }
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        const int slot = __float_as_int(place[s]);
        if (slot >= 0 && slot < K) {
            xi[slot] = ci[s];
            xd[slot] = cd[s];
        }
        if (slot >= 0) seen[seen_place(ci[s])] = ci[s];
    }
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        row.idx[s] = xi[lane + 64 * s];
        row.dist[s] = xd[lane + 64 * s];
    }
    row.refresh_tau();
    row.changed = true;
    return true;
}

// CL: 64 CL is at least the largest bucket.  The distances and ids of the next trees travel while the candidates of the
// present ones are offered.  (Ids requested only where a distance may still enter, a group later: 4 % slower at
// 400,000 x 100; what bounds the kernel is the issue of the insertions, not the bytes.)
template <int SL, int CL>
__global__ __launch_bounds__(256) void k_forest_merge(int N, int K, int T, const int* __restrict__ perm, const int2* __restrict__ info,
                                                      int pitch, const float* __restrict__ pair_dist, int* __restrict__ knn_idx,
                                                      float* __restrict__ knn_dist)
{
    constexpr int U = CL >= 4 ? 1 : 4 / CL;                 // trees of a group
    constexpr bool kRank = SL <= 2;
    __shared__ int seen_s[4][kSeen];
    __shared__ int xch_i[4][kRank ? 64 * SL : 1];
    __shared__ float xch_d[4][kRank ? 64 * SL : 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = (int)blockIdx.x * 4 + wave;
    if (p >= N) return;                                      // (a whole wavefront leaves)
    int* seen = seen_s[wave];
    const int2 where = lane < T ? info[(size_t)p * T + lane] : make_int2(0, 0);
    const size_t at = (size_t)p * (size_t)K;
    KnnRow<SL> row;
    row.load(knn_idx + at, knn_dist + at, K);
    auto request = [&](int j0, float (&dd)[U][CL], int (&cc)[U][CL]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = j0 + u;
            const int start = read_lane_i(where.x, j & 63), sm = read_lane_i(where.y, j & 63);
            const int m = sm & 0xffff, n = j < T ? sm >> 16 : 0;
            const size_t base = (size_t)j * (size_t)N + (size_t)start;
            const float* dr = pair_dist + (base + (size_t)m) * (size_t)pitch;
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                const int k = lane + 64 * v;
                const bool in = k < n && k != m;
                dd[u][v] = in ? dr[k] : INFINITY;
                cc[u][v] = in ? perm[base + k] : -1;
            }
        }
    };
    float da[U][CL], db[U][CL];
    int ca[U][CL], cb[U][CL];
    request(0, da, ca);
#pragma unroll
    for (int e = 0; e < kSeen / 64; ++e) seen[lane + 64 * e] = -1;
    wave_lds_sync();
#pragma unroll
    for (int s = 0; s < SL; ++s)
        if (row.idx[s] >= 0) seen[seen_place(row.idx[s])] = row.idx[s];
    wave_lds_sync();
    if constexpr (kRank) {
        bool fresh = small_bucket::fresh_row(row.idx[0], row.dist[0], p, min(K, 64));
        if (SL == 2) fresh = fresh && ballot64(row.idx[SL - 1] >= 0) == 0;
        if (fresh) {
            const int m = read_lane_i(where.y, 0) & 0xffff, n = read_lane_i(where.y, 0) >> 16;
            const bool self = read_lane_i(row.idx[0], 0) >= 0;
            const float self_d = read_lane_f(row.dist[0], 0);
            float dv[CL];
            int cv[CL];
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                const bool me = lane + 64 * v == m;
                dv[v] = me ? (self ? self_d : INFINITY) : da[0][v];
                cv[v] = me ? p : ca[0][v];
            }
            if (new_row_by_rank<SL, CL>(row, K, dv, cv, n, xch_i[wave], xch_d[wave], seen)) {
#pragma unroll
                for (int v = 0; v < CL; ++v) da[0][v] = INFINITY;        // done with
            }
        }
    }
    for (int j0 = 0; j0 < T; j0 += U) {
        request(j0 + U, db, cb);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                bool ok = row.enters(ca[u][v], da[u][v]);
                if (ballot64(ok) == 0) continue;
                const int h = seen_place(ca[u][v]);
                if (ok) ok = seen[h] != ca[u][v];
                if (ballot64(ok) == 0) continue;
                row.merge(ok, ca[u][v], da[u][v]);
                if (ok) seen[h] = ca[u][v];
                wave_lds_sync();
            }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int v = 0; v < CL; ++v) {
                da[u][v] = db[u][v];
                ca[u][v] = cb[u][v];
            }
    }
    if (row.changed) row.store(knn_idx + at, knn_dist + at);
}

int forest_pitch(int max_bucket) { return (max_bucket + 15) & ~15; }

}  // namespace

// May the buckets of several trees of this forest go together?  With fewer than four trees the chain of launches is
// too short to be worth it.  RSFK_FOREST_MERGE=1 / 0 says yes or no; a variable that asks for another form of the
// bucket step says no.
bool bucket_forest_wanted(int n_trees)
{
    const char* e = std::getenv("RSFK_FOREST_MERGE");
    if (e && *e) return e[0] == '1';
    for (const char* other : {"RSFK_BUCKET_SCREEN", "RSFK_GRAM_FROM", "RSFK_BUCKET_PAIRS"}) {
        const char* v = std::getenv(other);
        if (v && *v) return false;
    }
    return n_trees >= 4;
}

// Trees that go together (0: one tree after the other), out of n_trees.  Working memory: 2 GB, and it has to take two
// trees, or the K-NN rows travel as often as before.  Buckets of at most 72 points and rows of at most 64 neighbours
// have kernels of their own that skip most of a late tree's pairs; their chain of launches is the slower one up to about
// 200,000 points (time of the bucket step, one tree after the other -> together: 20,000 x 32, 50 trees 3.03 -> 0.31 ms,
// 150,000 x 100, 10 trees 1.61 -> 0.94, 250,000 x 20, K = 10, 40 trees 3.11 -> 3.28, 400,000 x 100, 50 trees
// 9.1 -> 9.8).  Larger buckets and longer rows gain at every size that fits (70,000 x 784, K = 90, 10 trees 5.0 -> 3.7), but for
// many trees over many points whose buckets fit into LDS whole and have far more points than a row has slots: there the later
// trees skip most pairs as well, and what the trees together move leaves the caches.  The line is at N sqrt(trees of the build) (largest bucket)
// / K^(3/4) = 31 million (1 + 1/D)^2, in the middle of what 664 builds of 2 to 64 dimensions, 6 to 60 trees, 200,000 to 2.5M points and buckets
// up to 73 .. 256 say (bucket step, one tree after the other / together): 210,000 x 4, K = 25, buckets of 50..200, 50 trees (27M) 8.2 / 5.3 ms;
// 210,000 x 2, K = 32, 64..256, 50 trees (28M) 12.8 / 6.2; 400,000 x 32, K = 32, 64..256, 12 trees (26M) 1.14 times, 50 trees (54M) 0.82;
// 400,000 x 2, K = 32, 64..256, 50 trees (54M; the line is at 70M) 18.0 / 12.0; 1M x 16, K = 16, 40..160, 6 trees (49M) 0.81, 50,
// K = 50, 64..256, 12 trees (47M) 1.07; 1.5M x 5, K = 7, 35..140, 26 trees (253M) 8.5 / 18.9.  With this line a step takes 0.6 % longer than the
// better form on (geometric) average, at worst 1.3 times; a line on N trees bucket / K took 3.7 %, at worst 2.4 times.
int bucket_forest_group(int N, int D, int K, int max_bucket, int n_trees, int all_trees)
{
    constexpr size_t kFloats = (size_t)1 << 29;
    constexpr int kMostPoints = 200000;
    if (max_bucket < 1 || max_bucket > 256) return 0;
    const char* e = std::getenv("RSFK_FOREST_MERGE");
    const bool forced = e && e[0] == '1';
    if (!forced && N > kMostPoints && K <= 64 && max_bucket <= medium_bucket_cap()) return 0;
    if (!forced && N > kMostPoints && K <= 64 && max_bucket <= bucket_rows_cap(D, K) &&
        N * std::sqrt((double)all_trees) * max_bucket >= 3.1e7 * (1.0 + 1.0 / D) * (1.0 + 1.0 / D) * std::pow((double)K, 0.75))
        return 0;
    const int group = (int)std::min<size_t>((size_t)std::min(n_trees, 64), kFloats / ((size_t)N * (size_t)forest_pitch(max_bucket)));
    return group >= std::min(2, n_trees) ? group : 0;
}

size_t bucket_forest_floats(int N, int max_bucket, int n_trees)
{
    return (size_t)N * (size_t)forest_pitch(max_bucket) * (size_t)n_trees;
}

// Buckets of T trees (perm: T x N, leaf tables and stats of those trees) into the K-NN rows.  most_blocks: the largest
// number of buckets of at most kBucketSplit points, plus tri times the larger ones, of any of the trees.
int launch_bucket_knn_forest(const float* points, int N, int D, int K, int T, const int* perm, const int* leaf_start, const int* leaf_size,
                             int leaf_cap, const int* stats, const int* host_stats, int max_bucket, float* pair_dist, int* info,
                             int* knn_idx, float* knn_dist, hipStream_t stream)
{
    RSFK_CHECK(K >= 1 && K <= kMaxK && T >= 1 && T <= 64 && max_bucket <= 256, "bucket K-NN of a forest: out of range");
    const int max_tiles = (max_bucket + kTile - 1) / kTile, tri = max_tiles * (max_tiles + 1) / 2;
    int most = 1;
    for (int j = 0; j < T; ++j) {
        const int n_big = host_stats[5 * j + 4], n_small = host_stats[5 * j] - n_big;
        most = std::max(most, n_small + n_big * tri);
    }
    const int pitch = forest_pitch(max_bucket);
    int2* where = reinterpret_cast<int2*>(info);
    hipLaunchKernelGGL(k_forest_pairs, dim3((unsigned)most, (unsigned)T), dim3(256), 0, stream, points, N, D, T, perm, leaf_start,
                       leaf_size, leaf_cap, stats, max_tiles, tri, pitch, pair_dist, where);
    const dim3 grid((unsigned)((N + 3) / 4)), block(256);
#define RSFK_FOREST_CASE(SLV)                                                                                               \
    do {                                                                                                                    \
        if (max_bucket <= 64)                                                                                               \
            hipLaunchKernelGGL((k_forest_merge<SLV, 1>), grid, block, 0, stream, N, K, T, perm, where, pitch, pair_dist,     \
                               knn_idx, knn_dist);                                                                          \
        else if (max_bucket <= 128)                                                                                         \
            hipLaunchKernelGGL((k_forest_merge<SLV, 2>), grid, block, 0, stream, N, K, T, perm, where, pitch, pair_dist,     \
                               knn_idx, knn_dist);                                                                          \
        else                                                                                                                \
            hipLaunchKernelGGL((k_forest_merge<SLV, 4>), grid, block, 0, stream, N, K, T, perm, where, pitch, pair_dist,     \
                               knn_idx, knn_dist);                                                                          \
    } while (0)
    switch (row_slots(K)) {
    case 1: RSFK_FOREST_CASE(1); break;
    case 2: RSFK_FOREST_CASE(2); break;
    case 4: RSFK_FOREST_CASE(4); break;
    case 8: RSFK_FOREST_CASE(8); break;
    default: RSFK_FOREST_CASE(16); break;
    }
#undef RSFK_FOREST_CASE
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
