// Neighbourhood exploration: every point looks at the neighbours of its
// neighbours (taken from a snapshot of the index array) and merges the closer
// ones into its own row.  Replaces nearest_neighbors_exploring
// (src/kernels/nearest_neighbors_exploring.cu:41-146) and its host loop
// (src/rsfk.cu:2100-2135).
//
// One wavefront per point, in three stages:
//
//  1. collect.  The K*K candidate ids are read with coalesced row reads of the
//     snapshot (16 rows of 64 ids in flight at a time) and put into a hash set in
//     LDS that was seeded with the point itself and its current row.  Only ids
//     that are new to the set survive, so each distinct candidate is looked at
//     once.  (The reference re-evaluates repeats; the result is the same because
//     a rejected candidate stays rejected -- the row maximum only decreases -- and
//     an accepted one is found in the row afterwards.)  The set is then compacted
//     in place into the list of candidates.  When the set cannot hold all K*K ids
//     (large K) the neighbours are processed in groups, each with a fresh set.
//
//  2. screen, on the bfloat16 copy of the points.  64 candidates at a time: their
//     rows (up to 128 dimensions = 256 bytes each) are requested with coalesced
//     128-byte segments, 8 lanes per row, while the previous 64 are being
//     evaluated (two batches of loads are in flight per wavefront: the stage is
//     bound by gather latency, so memory-level parallelism is what counts).  Rows
//     are transposed through LDS and each lane accumulates for "its" candidate
//     the approximate squared distance d~ and the quantity T below; a candidate
//     with d~ - E >= row maximum cannot enter the row and is dropped without its
//     fp32 row ever being touched.
//
//  3. exact.  The few candidates that pass get the exact distance from the fp32
//     rows (same gather/transposition, sequential fused multiply-add chain per
//     candidate: the arithmetic of the bucket kernel, compute_knn_from_buckets.cu:40-54,
//     so a pair has one distance value everywhere) and are offered to the sorted row.
//
// Error bound of the screen.  bfloat16 keeps 8 significant bits, so c~ = c + e with
// |e_d| <= 2^-8 |c_d| <= 2^-8 (1+2^-7) |c~_d| (round to nearest).  From
// (x-c)^2 = (x-c~)^2 + 2(x-c~)e + e^2:
//     |d~ - d| <= 2^-7 (1+2^-7) T + 2^-16 (1+2^-6) Q,   T = sum |x_d - c~_d| |c~_d|,  Q = sum c~_d^2.
// Both fp32 sums (d~ here, d in the exact path) are sums of non-negative terms, so
// each is within D 2^-24 (relative) of its real value.  E below is larger than the
// total; Q comes precomputed with the copy.
#include "rsfk_common.hpp"
#include "knn_list.hpp"
#include "forest.hpp"
#include "exact_batch.hpp"
#include "join_bounds.hpp"
#include <algorithm>

namespace rsfk {

namespace {

constexpr int kPitch = kChunk + 4;      // 36 words = 9 x 16 B: conflict-free b128 reads down a column of rows
constexpr int kBlockB = 128;            // bfloat16 dimensions per pipeline stage of the screen (2 x 64)
constexpr int kQueue2 = 128;            // candidates waiting for the exact distance
constexpr int kIdRows = 16;             // batches of 64 candidate ids loaded back to back
constexpr int kEmpty = (int)0x80000000; // free slot of the hash set

__device__ __forceinline__ uint32_t hash_id(int c)
{
    uint32_t h = (uint32_t)c * 0x9E3779B1u;
    return h ^ (h >> 15);
}

// Set of ids with open addressing.  Seeds (ids that must not become candidates) are
// stored as -id-1, candidates as id.  Returns true when c was new.  The caller
// guarantees a free slot exists.
__device__ __forceinline__ bool set_insert(int* table, int mask, int c, bool seed)
{
    uint32_t h = hash_id(c) & (uint32_t)mask;
    const int stored = seed ? -c - 1 : c;
    for (int i = 0; i <= mask; ++i) {
        const int old = atomicCAS(&table[h], kEmpty, stored);
        if (old == kEmpty) return true;
        if (old == c || old == -c - 1) return false;
        h = (h + 1) & (uint32_t)mask;
    }
    return false;
}

// The same for a candidate, returning its place in the table (whether new or already there), or -1 when the id is a
// seed (or the table is full).
__device__ __forceinline__ int set_insert_at(int* table, int mask, int c)
{
    uint32_t h = hash_id(c) & (uint32_t)mask;
    for (int i = 0; i <= mask; ++i) {
        const int old = atomicCAS(&table[h], kEmpty, c);
        if (old == kEmpty || old == c) return (int)h;
        if (old == -c - 1) return -1;
        h = (h + 1) & (uint32_t)mask;
    }
    return -1;
}

__device__ __forceinline__ void screen_pair(uint32_t w, float x0, float x1, float& da, float& ta)
{
    const float c0 = __uint_as_float(w << 16);
    const float c1 = __uint_as_float(w & 0xffff0000u);
    const float f0 = x0 - c0, f1 = x1 - c1;
    da = __builtin_fmaf(f0, f0, da);
    da = __builtin_fmaf(f1, f1, da);
    ta = __builtin_fmaf(fabsf(f0), fabsf(c0), ta);
    ta = __builtin_fmaf(fabsf(f1), fabsf(c1), ta);
}

// One pipeline stage of the screen = 128 bfloat16 dimensions of 64 candidate rows.
struct ScreenLoads {
    uint4 v[16];             // v[h*8+i]: half h (64 dimensions), rows i*8+sub, piece lane&7
};

__device__ __forceinline__ void screen_issue(ScreenLoads& S, const int* list, int n, const uint16_t* __restrict__ rows,
                                             int Db, int Dv, int b0)
{
    const int lane = lane_id();
    const int sub = lane >> 3, piece = lane & 7;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = i * 8 + sub;
        const uint16_t* rp = rows + (size_t)list[r < n ? r : 0] * (size_t)Db + b0 + piece * 8;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            S.v[h * 8 + i] = make_uint4(0, 0, 0, 0);
            if (b0 + h * 64 + piece * 8 < Dv) S.v[h * 8 + i] = *reinterpret_cast<const uint4*>(rp + h * 64);
        }
    }
}

// Accumulate one stage into (da, ta) of this lane's candidate.
__device__ __forceinline__ void screen_consume(const ScreenLoads& S, const ExploreLds& L, int Db, int b0, float& da,
                                               float& ta)
{
    const int lane = lane_id();
    const int sub = lane >> 3, piece = lane & 7;
    uint32_t* tile = reinterpret_cast<uint32_t*>(L.tile);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int d0 = b0 + h * 64;
        if (d0 >= Db) break;
        wave_lds_sync();                 // previous reads of the tile are done
#pragma unroll
        for (int i = 0; i < 8; ++i)
            *reinterpret_cast<uint4*>(&tile[(i * 8 + sub) * kPitch + piece * 4]) = S.v[h * 8 + i];
        wave_lds_sync();
        const int pieces = min(8, (Db - d0) >> 3);
        const uint32_t* mine = &tile[lane * kPitch];
        const float* xs = &L.xrow[d0];
        for (int q = 0; q < pieces; ++q) {
            const uint4 w = *reinterpret_cast<const uint4*>(mine + 4 * q);
            const float4 xa = *reinterpret_cast<const float4*>(xs + 8 * q);
            const float4 xb = *reinterpret_cast<const float4*>(xs + 8 * q + 4);
            screen_pair(w.x, xa.x, xa.y, da, ta);
            screen_pair(w.y, xa.z, xa.w, da, ta);
            screen_pair(w.z, xb.x, xb.y, da, ta);
            screen_pair(w.w, xb.z, xb.w, da, ta);
        }
    }
}

// Count of the exact distances of a launch, for the report of a build: one addition per wavefront, to one of 256
// slots a cache line apart (stat may be null).
__device__ __forceinline__ void count_exact(unsigned long long* stat, int n)
{
    if (stat && n > 0 && lane_id() == 0) atomicAdd(&stat[32 * (blockIdx.x & 255)], (unsigned long long)n);
}

// Stages are numbered s = batch * nblk + block; list holds U candidates.
struct ScreenCtx {
    const int* list;
    int U, nblk, Db, Dv, D;
};

template <int SL>
__device__ __forceinline__ void screen_stage_finish(const ScreenCtx& C, const ExploreLds& L, const Bf16Copy& bf, int batch,
                                                    float da, float ta, KnnRow<SL>& row, int& queued2,
                                                    const float* __restrict__ points, bool vec_ok, int& n_exact)
{
    const int lane = lane_id();
    const int n = min(64, C.U - batch * 64);
    const int my_c = C.list[batch * 64 + (lane < n ? lane : 0)];
    const float qn = bf.norms[my_c];
    const float slack = (float)(C.D + 8) * (1.0f / 4194304.0f);      // (D+8) 2^-22: fp32 summation error of both sums
    const float e = ta * (1.02f / 128.0f) + qn * (1.05f / 65536.0f) + da * slack;
    const bool may = lane < n && (da - e <= row.tau);
    const uint64_t pm = ballot64(may);
    if (pm == 0) return;
    if (may) L.queue2[queued2 + mask_prefix(pm)] = my_c;
    queued2 += __popcll(pm);
    if (queued2 >= 64) {
        wave_lds_sync();
        exact_batch<SL>(L, L.queue2, 64, points, C.D, vec_ok, row);
        n_exact += 64;
        const int rest = queued2 - 64;
        const int mv = lane < rest ? L.queue2[64 + lane] : 0;
        wave_lds_sync();
        if (lane < rest) L.queue2[lane] = mv;
        queued2 = rest;
        wave_lds_sync();
    }
}

template <int SL>
__device__ __forceinline__ void screen_all(const ScreenCtx& C, const ExploreLds& L, const Bf16Copy& bf, KnnRow<SL>& row,
                                           int& queued2, const float* __restrict__ points, bool vec_ok, int& n_exact)
{
    const int nb = (C.U + 63) >> 6;
    const int stages = nb * C.nblk;
    ScreenLoads A, B;
    float da = 0.0f, ta = 0.0f;
    auto issue = [&](ScreenLoads& S, int s) {
        const int batch = s / C.nblk, blk = s - batch * C.nblk;
        screen_issue(S, C.list + batch * 64, min(64, C.U - batch * 64), bf.rows, C.Db, C.Dv, blk * kBlockB);
    };
    auto consume = [&](const ScreenLoads& S, int s) {
        const int batch = s / C.nblk, blk = s - batch * C.nblk;
        if (blk == 0) { da = 0.0f; ta = 0.0f; }
        screen_consume(S, L, C.Dv, blk * kBlockB, da, ta);
        if (blk == C.nblk - 1) screen_stage_finish<SL>(C, L, bf, batch, da, ta, row, queued2, points, vec_ok, n_exact);
    };
    if (stages > 0) issue(A, 0);
    for (int s = 0; s < stages; s += 2) {
        if (s + 1 < stages) issue(B, s + 1);
        consume(A, s);
        if (s + 1 < stages) {
            if (s + 2 < stages) issue(A, s + 2);
            consume(B, s + 1);
        }
    }
}

template <int SL, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_explore(const float* __restrict__ points, Bf16Copy bf, int N, int D, int K,
                                                         const int* __restrict__ old_idx, int* __restrict__ knn_idx,
                                                         float* __restrict__ knn_dist, int table_size, int wave_lds_ints,
                                                         int dpad, int rows_per_group, const int* __restrict__ todo,
                                                         int first, int n_todo, unsigned long long* __restrict__ stat)
{
    extern __shared__ __align__(16) int lds_i[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int slot = first + blockIdx.x * WAVES + wave;
    if (slot >= (todo ? n_todo : N)) return;              // whole wavefront leaves together
    const int p = todo ? todo[slot] : slot;               // all points, or the listed ones
    int* base = lds_i + (size_t)wave * (size_t)wave_lds_ints;
    ExploreLds L;
    L.tile = reinterpret_cast<float*>(base);                        // 64*kPitch words, 16-byte aligned
    L.xrow = reinterpret_cast<float*>(base + 64 * kPitch);          // dpad floats (multiple of 8)
    L.queue2 = base + 64 * kPitch + dpad;
    L.table = L.queue2 + kQueue2;
    L.srow = L.table + table_size;
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);
    const bool use_screen = bf.rows != nullptr;
    const int mask = table_size - 1;

    KnnRow<SL> row;
    row.load(knn_idx + (size_t)p * K, knn_dist + (size_t)p * K, K);
    for (int k = lane; k < K; k += 64) L.srow[k] = old_idx[(size_t)p * K + k];
    const float* xp = points + (size_t)p * D;
    for (int d = lane; d < dpad; d += 64) L.xrow[d] = d < D ? xp[d] : 0.0f;

    ScreenCtx C;
    C.list = L.table;
    C.Db = bf16_pitch(D);
    C.Dv = bf16_valid(D);
    C.D = D;
    C.nblk = (C.Dv + kBlockB - 1) / kBlockB;
    int queued2 = 0;                                       // wave-uniform
    int n_exact = 0;                                       // exact distances of this point (wave-uniform)

    for (int i0 = 0; i0 < K; i0 += rows_per_group) {
        const int i1 = min(K, i0 + rows_per_group);
        // ---- collect -----------------------------------------------------------------
        wave_lds_sync();
        for (int i = lane; i < table_size; i += 64) L.table[i] = kEmpty;
        wave_lds_sync();
        if (lane == 0) set_insert(L.table, mask, p, true);
#pragma unroll
        for (int s = 0; s < SL; ++s)
            if (row.idx[s] >= 0) set_insert(L.table, mask, row.idx[s], true);
        const int e_begin = i0 * K, e_end = i1 * K;
        for (int g0 = e_begin; g0 < e_end; g0 += 64 * kIdRows) {
            int cand[kIdRows];
#pragma unroll
            for (int b = 0; b < kIdRows; ++b) {
                const int e = g0 + b * 64 + lane;
                int c = -1;
                if (e < e_end) {
                    const int i = e / K, k = e - i * K;
                    const int q = L.srow[i];
                    if (q >= 0 && q < N) c = old_idx[(size_t)q * K + k];
                }
                cand[b] = c;
            }
#pragma unroll
            for (int b = 0; b < kIdRows; ++b) {
                if (g0 + b * 64 >= e_end) break;
                const int c = cand[b];
                if (c >= 0 && c < N) set_insert(L.table, mask, c, false);
            }
        }
        wave_lds_sync();
        // ---- compact the set in place into the candidate list --------------------------
        int U = 0;
        for (int t0 = 0; t0 < table_size; t0 += 64) {
            const int v = L.table[t0 + lane];
            const bool is_cand = v >= 0;
            const uint64_t m = ballot64(is_cand);
            wave_lds_sync();             // all reads of this block are done before the front is overwritten
            if (is_cand) L.table[U + mask_prefix(m)] = v;
            U += __popcll(m);
        }
        wave_lds_sync();
        C.U = U;
        // ---- screen / exact ------------------------------------------------------------
        if (use_screen) {
            screen_all<SL>(C, L, bf, row, queued2, points, vec_ok, n_exact);
        } else {
            for (int off = 0; off < U; off += 64) {
                wave_lds_sync();
                exact_batch<SL>(L, L.table + off, min(64, U - off), points, D, vec_ok, row);
            }
            n_exact += U;
        }
    }
    // drain the second queue (at most 127 entries)
    for (int off = 0; off < queued2; off += 64) {
        wave_lds_sync();
        exact_batch<SL>(L, L.queue2 + off, min(64, queued2 - off), points, D, vec_ok, row);
    }
    n_exact += queued2;
    count_exact(stat, n_exact);
    if (row.changed) row.store(knn_idx + (size_t)p * K, knn_dist + (size_t)p * K);
}

// Number of entry (p, k) of the graph snapshot, p K + k, or -1 when the slot holds no valid neighbour (the join writes
// nothing for such an entry).
__device__ __forceinline__ int graph_entry(const int* __restrict__ old_idx, int N, int K, int p, int k)
{
    const int q = old_idx[(size_t)p * K + k];
    return q >= 0 && q < N ? p * K + k : -1;
}

constexpr int kMergeChunk = 16;
// up to this many candidates of a point are evaluated without a look at their codes
constexpr int kFewCandidates = 32;
// 16-byte pieces of a candidate's row a lane requests from the tile together (exact_batch): 16 dimensions per wait for
// LDS.  (Measured: 1M x 256 pass 26.2 -> 24.8 ms, 70k x 784 pass 26.2 -> 25.0 ms; eight pieces cost the workgroup
// kernel its second wavefront per SIMD: 39 ms.)
constexpr int kChainGroup = 4;
constexpr int kMergeTile = 64 * (kMergeChunk + 4);
// Short rows are read by the lane that runs their chain, 32 dimensions at a time, without the transposing tile in LDS
// (exact_direct): the LDS of a wavefront shrinks by the tile.  This is the size of a wavefront's memory that the launches are
// planned with; what a launch then takes is merge_direct's choice.
__host__ __device__ inline int merge_tile_ints(int dpad, int direct_max) { return dpad <= direct_max ? 0 : kMergeTile; }
__host__ __device__ inline int merge_rank_at(int table, int K, bool with_bounds)
{
    return table + ((K + 3) & ~3) + (with_bounds ? table / 4 * 7 : 0);
}
int merge_direct_env()
{
    static const int v = [] {
        const char* e = std::getenv("RSFK_MERGE_DIRECT");
        return e ? std::atoi(e) : -1;
    }();
    return v;
}
int merge_direct_max() { return merge_direct_env() >= 0 ? merge_direct_env() : 128; }
// Does a launch read rows of this many dimensions without the tile?  With all candidates of a point to be evaluated the trips to
// memory of a long row weigh more than the wavefronts that the tile's 5 KB keep out (measured: 1M x 100 merge 4.4 -> 3.4 ms without,
// 10M x 32 43 -> 27 ms, 1M x 256 slower), hence 128.  Where the join's codes leave a point few of them, most lanes of the tile's
// loads carry nothing and the wavefronts count for longer: whole pass at 1M x 256, K = 32 in clusters 15.5 -> 14.0 ms, 500k x 132
// 5.97 -> 4.98, 150k x 280, K = 44 4.65 -> 4.15; 150k x 320, K = 33 3.98 -> 4.24, x 384, K = 36 4.93 -> 5.18: 288.  Rows that are not
// in whole 16-byte pieces take four times the loads: 150k x 161, K = 16 1.23 -> 1.18, x 231 1.41 -> 1.48, x 255 1.45 -> 1.58: 192.
constexpr int kDirectCoded = 288, kDirectCodedOdd = 192;
bool merge_direct(int D, int dpad, bool coded)
{
    if (!coded || merge_direct_env() >= 0) return dpad <= merge_direct_max();
    return dpad <= ((D & 3) == 0 ? kDirectCoded : kDirectCodedOdd);
}

// Rows of the candidates by four lanes in turn (exact_direct) or by a lane each?  The former saves requests, and takes instructions for lanes that have no
// candidate too: it needs long rows and many candidates, and where codes leave a point few of them, points beyond the last cache (256 MB) as well.  Merge,
// own -> quads: without codes, 100,000 points, K = 10 x 128 177 -> 219 us, K = 12 x 100 167 -> 209, K = 16 x 40 137 -> 156, x 96 210 -> 203 (1M 1.97 -> 2.06 ms), x 128
// 293 -> 241, 755,473 x 115 (sparse) 2.97 -> 1.95 ms, 1M x 112, 10 trees 1.86 -> 2.18, K = 18 x 64 188 -> 178, K = 20 x 40 180 -> 181, x 48 198 -> 184 (1M 1.83 -> 1.78), x 64 239 -> 194, K = 24 x 28 207 -> 192, x 48 290 -> 233, K = 32 x 20 282 -> 296,
// x 24 305 -> 295 (1M 2.46 -> 2.24), x 36 441 -> 364, K = 45 x 12 507 -> 539, x 24 611 -> 600, x 40 939 -> 766; 1M x 100, K = 32 6.41 -> 4.52 ms.  With codes, K = 8, 300,000 x 256
// 0.82 -> 1.11 ms, K = 16, 20,000 x 208 78 -> 95 us, K = 24, 1M x 208 4.83 -> 5.26, K = 28, 1M x 256 5.86 -> 5.90, K = 32, 300,000 x 132 1.38 -> 1.52, x 256 1.93 -> 1.98, 450,000 x 288
// 3.15 -> 3.03, 1M x 132 4.35 -> 4.67, x 160 4.56 -> 4.76, x 208 5.72 -> 5.62, x 256 5.92 -> 5.61, x 288 7.18 -> 6.74.
// (RSFK_MERGE_QUADS=0|1: never, always)
bool merge_quads(int N, int D, int K, bool coded)
{
    const char* e = std::getenv("RSFK_MERGE_QUADS");
    if (e && *e) return e[0] == '1';
    if (coded) return K >= 32 && D > 200 && (size_t)N * (size_t)D >= (size_t)1 << 27;
    return (K >= 24 && D >= 24) || (K >= 18 && D >= 48) || (K >= 16 && D >= 96);
}

// Exploration of the points whose candidates the join has marked (explore_join.hip): entry (p, k) of
// the graph has the mask of neighbour slots at pass[p K + k] (entries without a valid neighbour have none).  One wavefront per point: gather
// the marked ids, drop repeats and ids the row holds (hash set), exact distances, merge.  Points with
// more marks than the LDS of this launch takes are appended to todo_out (for a launch with more LDS
// per wavefront, or for the general kernel; share > 0: to the point's share of it, explore_ws_share_lists).  todo_in: the points to work on,
// or null for all.  Per-wavefront LDS (ints): with the tile tile[64*20] | xrow[dpad] | table[table_size] | srow[K] | marked[3/4 table_size]
// | with codes: tbound[table_size] | without the tile: the ranks (merge_rank_at).
// kFormTile: the candidates' rows go through the transposing tile (not merge_direct); kFormOwn: a lane reads its candidate's row; kFormDirect, kFormDirectCoded: four
// lanes read rows in turn (exact_direct, merge_quads), without and with codes.  The forms are kernels of their own, so that none carries
// the registers of another: by quads and without codes 75, held to the 72 of seven wavefronts per SIMD (two are spilled, 12 bytes of scratch a lane), with codes
// 85, held to the 80 of six (10M x 32 17.33 ms, 17.98 with six wavefronts, 24.2 with the 99 registers of code of its own choice; 1M x 256 5.65, 6.33 with seven).
enum { kFormTile, kFormOwn, kFormDirect, kFormDirectCoded };
template <int SL, int WAVES, int FORM>
__global__ __launch_bounds__(64 * WAVES, FORM == kFormTile || FORM == kFormOwn || SL > 1 ? 1 : FORM == kFormDirect ? 7 : 6) void k_explore_merge(const float* __restrict__ points, int N, int D, int K,
                                                               const int* __restrict__ old_idx, int* __restrict__ knn_idx,
                                                               float* __restrict__ knn_dist, int table_size,
                                                               int wave_lds_ints, int dpad,
                                                               const uint32_t* __restrict__ pass, JoinBounds jb,
                                                               const int* __restrict__ todo_in, int n_in,
                                                               int* __restrict__ todo_out, int share, int* __restrict__ n_out,
                                                               unsigned long long* __restrict__ stat,
                                                               const int* __restrict__ order)
{
    extern __shared__ __align__(16) int lds_m[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int slot = die_local_place(blockIdx.x, gridDim.x) * WAVES + wave;
    if (slot >= (todo_in ? n_in : N)) return;             // whole wavefront leaves together
    const int p = todo_in ? todo_in[slot] : (order ? order[slot] : slot);
    const int MW = (K + 31) >> 5;
    int* base = lds_m + (size_t)wave * (size_t)wave_lds_ints;
    // Rows of at most 64 neighbours (one slot per lane): everything the point needs from memory before its candidates
    // are known -- its K-NN row, the snapshot of its neighbours, its mark words, its coordinates -- is requested at once;
    // none of these addresses depends on another's data.  (Longer rows: one after the other, as they are needed.)
    constexpr bool kEarly = SL == 1, TILE = FORM == kFormTile;
    KnnRow<SL> row;
    int q_own = -1;
    uint32_t pw[2] = {0u, 0u};
    if (kEarly) {
        const size_t at = (size_t)p * K + (lane < K ? lane : 0);
        row.idx[0] = knn_idx[at];
        row.dist[0] = knn_dist[at];
        q_own = old_idx[at];
        pw[0] = pass[at * MW];
        if (MW > 1) pw[1] = pass[at * MW + 1];
        const float* xp0 = points + (size_t)p * D;
        float* xr = reinterpret_cast<float*>(base + (TILE ? kMergeTile : 0));
        for (int d = lane; d < dpad; d += 64) xr[d] = d < D ? xp0[d] : 0.0f;
        if (lane >= K) { row.idx[0] = -2; row.dist[0] = INFINITY; q_own = -1; }
        if (!(q_own >= 0 && q_own < N)) { pw[0] = 0u; pw[1] = 0u; }          // the join writes nothing for such an entry
    }
    int bits = 0;
    if (kEarly) {
        bits = __popc(pw[0]) + __popc(pw[1]);
    } else {
        for (int k = lane; k < K; k += 64) {
            const int j = graph_entry(old_idx, N, K, p, k);
            if (j >= 0)
                for (int w = 0; w < MW; ++w) bits += __popc(pass[(size_t)j * MW + w]);
        }
    }
    const int n_given = wave_sum_i(bits);
    if (n_given == 0) return;
    if (n_given + K + 1 > table_size / 4 * 3) {
        const int s = share > 0 ? slot % kTodoShares : 0;
        if (lane == 0) todo_out[(size_t)s * (size_t)share + (size_t)atomicAdd(n_out + 32 * s, 1)] = p;
        return;
    }
    ExploreLds L;
    L.tile = reinterpret_cast<float*>(base);
    constexpr int tile_ints = TILE ? kMergeTile : 0;
    L.xrow = reinterpret_cast<float*>(base + tile_ints);
    L.queue2 = nullptr;
    L.table = base + tile_ints + dpad;
    L.srow = L.table + table_size;
    const uint16_t* __restrict__ bounds = FORM == kFormDirect ? nullptr : jb.codes;
    // with bounds: the code of the id in the same place of the set, behind the list of marks
    int* tbound = bounds ? L.srow + K + table_size / 4 * 3 : nullptr;
    // without the tile: the ranks' working memory, in place of the list of marks or behind the bounds
    if (!TILE) L.rank = reinterpret_cast<double*>(base + dpad + merge_rank_at(table_size, K, bounds != nullptr));
    const int KP = (K + 31) & ~31;
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);

    if (kEarly) {
        row.init_from_regs(K);
        if (lane < K) L.srow[lane] = q_own;
    } else {
        row.load(knn_idx + (size_t)p * K, knn_dist + (size_t)p * K, K);
        for (int k = lane; k < K; k += 64) L.srow[k] = old_idx[(size_t)p * K + k];
        const float* xp = points + (size_t)p * D;
        for (int d = lane; d < dpad; d += 64) L.xrow[d] = d < D ? xp[d] : 0.0f;
    }

    int ts = 64;
    while (ts < 2 * (n_given + K + 1)) ts <<= 1;
    ts = min(ts, table_size);
    const int mask = ts - 1;
    for (int i = lane; i < ts; i += 64) {
        L.table[i] = kEmpty;
        if (tbound) tbound[i] = 0x7fffffff;
    }
    wave_lds_sync();
    if (lane == 0) set_insert(L.table, mask, p, true);
#pragma unroll
    for (int s = 0; s < SL; ++s)
        if (row.idx[s] >= 0) set_insert(L.table, mask, row.idx[s], true);
    // list of the marked (neighbour, slot) pairs, so that the ids can be gathered by all lanes at once
    // instead of one after the other per neighbour
    int* marked = L.srow + K;
    int n_marked = 0;                                     // wave-uniform
    for (int k0 = 0; k0 < K; k0 += 64) {
        const int k = k0 + lane;
        const int j = kEarly ? (q_own >= 0 && q_own < N ? p * K + k : -1) : (k < K ? graph_entry(old_idx, N, K, p, k) : -1);
        int mine = 0;
        if (kEarly) mine = bits;
        else if (j >= 0)
            for (int w = 0; w < MW; ++w) mine += __popc(pass[(size_t)j * MW + w]);
        int at = n_marked + wave_excl_scan_i(mine);
        if (j >= 0) {
            for (int w = 0; w < MW; ++w) {
                uint32_t m = kEarly ? pw[w & 1] : pass[(size_t)j * MW + w];
                while (m) {
                    const int b = __ffs(m) - 1;
                    m &= m - 1;
                    marked[at++] = k | ((32 * w + b) << 8);
                }
            }
        }
        n_marked += wave_sum_i(mine);
    }
    wave_lds_sync();
    // (the ids of 256 marks are requested together: a point's marks then cost one trip to memory, not one per 64)
    for (int i0 = 0; i0 < n_marked; i0 += 256) {
        int c[4], lb[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int i = i0 + 64 * u + lane;
            c[u] = -1;
            lb[u] = 0;
            if (i < n_marked) {
                const int e = marked[i];
                c[u] = old_idx[(size_t)L.srow[e & 255] * K + (e >> 8)];
                // the join's code of the pair: entry p K + k of the graph, column = slot in the neighbour's row
                if (bounds) lb[u] = bounds[((size_t)p * K + (e & 255)) * (size_t)KP + (e >> 8)];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (c[u] >= 0 && c[u] < N) {
                if (tbound) {
                    const int at = set_insert_at(L.table, mask, c[u]);
                    if (at >= 0) atomicMin(&tbound[at], lb[u]);
                } else {
                    set_insert(L.table, mask, c[u], false);
                }
            }
        }
    }
    wave_lds_sync();
    // compact the set in place into the candidate list (and the bounds with it)
    int U = 0;
    for (int t0 = 0; t0 < ts; t0 += 64) {
        const int v = L.table[t0 + lane];
        const int vb = tbound ? tbound[t0 + lane] : 0;
        const bool is_cand = v >= 0;
        const uint64_t m = ballot64(is_cand);
        wave_lds_sync();
        if (is_cand) {
            L.table[U + mask_prefix(m)] = v;
            if (tbound) tbound[U + mask_prefix(m)] = vb;
        }
        U += __popcll(m);
    }
    wave_lds_sync();
    int n_exact = 0;                                      // exact distances of this point (wave-uniform)
    float reach = INFINITY;                               // what the row's last slot will be at most
    auto batch = [&](const int* list, int n) {
        n_exact += n;
        if (!TILE) exact_direct<SL, FORM != kFormOwn, true>(L, list, n, points, D, vec_ok, row, reach);
        else exact_batch<SL, kMergeChunk, true, kChainGroup, true>(L, list, n, points, D, vec_ok, row, reach);    // two steps of gathers in flight
    };
    if (tbound == nullptr || U <= kFewCandidates) {
        for (int off = 0; off < U; off += 64) {
            wave_lds_sync();
            batch(L.table + off, min(64, U - off));
        }
    } else {
        // The reach of the row: the smallest upper end of a code at or below which the row and its candidates have K entries.
        // (The candidates are distinct and not in the row.  Codes of 0 have no upper end.)
        const CodeReader codes(jb, p);
        {
            constexpr int kIn = 4;                        // steps of 64 candidates whose codes stay in registers
            int cc[kIn], rc[SL];
#pragma unroll
            for (int u = 0; u < kIn; ++u) {
                const int b = 64 * u + lane < U ? tbound[64 * u + lane] : 0;
                cc[u] = b > 0 ? b : kCodeTop;
            }
#pragma unroll
            for (int s = 0; s < SL; ++s) rc[s] = codes.code_of(row.dist[s]);
            int lo = 1, hi = kCodeTop;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                int n = 0;
#pragma unroll
                for (int u = 0; u < kIn; ++u) n += __popcll(ballot64(cc[u] <= mid));
                for (int t0 = 64 * kIn; t0 < U; t0 += 64) {
                    const int b = t0 + lane < U ? tbound[t0 + lane] : 0;
                    n += __popcll(ballot64(b > 0 && b <= mid));
                }
#pragma unroll
                for (int s = 0; s < SL; ++s) n += __popcll(ballot64(rc[s] <= mid));
                if (n >= K) hi = mid;
                else lo = mid + 1;
            }
            if (lo < kCodeTop) reach = codes.reach(lo);
        }
        // What is beyond it is never read.  What is left goes in rounds, nearer bounds first: a round takes the candidates whose bound
        // is not above the row's last slot (it shrinks from round to round) and -- while more than a batch of them is left -- not above
        // the mean of these bounds.  The ids of a round are gathered in the list of marks, which is no longer needed.
        constexpr int kDone = 0x7fffffff;
        int* round_ids = marked;
        while (true) {
            const int last = codes.last_code(fminf(row.tau, reach));
            int n_el = 0, sum = 0;
            for (int t0 = 0; t0 < U; t0 += 64) {
                const int b = t0 + lane < U ? tbound[t0 + lane] : kDone;
                const bool el = b <= last;
                n_el += __popcll(ballot64(el));
                sum += el ? b : 0;
            }
            if (n_el == 0) break;
            sum = wave_sum_i(sum);
            const int cut = n_el <= 64 ? last : min(last, sum / n_el);  // (the smallest bound is never above the mean)
            int n_round = 0;
            for (int t0 = 0; t0 < U; t0 += 64) {
                const int b = t0 + lane < U ? tbound[t0 + lane] : kDone;
                const bool take = b <= cut;
                const uint64_t m = ballot64(take);
                if (take) {
                    round_ids[n_round + mask_prefix(m)] = L.table[t0 + lane];
                    tbound[t0 + lane] = kDone;
                }
                n_round += __popcll(m);
            }
            for (int off = 0; off < n_round; off += 64) {
                wave_lds_sync();
                batch(round_ids + off, min(64, n_round - off));
            }
            wave_lds_sync();
        }
    }
    count_exact(stat, n_exact);
    if (row.changed) row.store(knn_idx + (size_t)p * K, knn_dist + (size_t)p * K);
}

// The same for rows so long that the set of one point takes much of a wavefront's LDS (K >= 64, or 32 with codes, launch_explore:
// a point has up to K^2 marks): one workgroup of four wavefronts per point.
//
// A candidate can only end up in the row if its exact distance is at most the row's last slot at the end, and every exact distance is
// a whole fp32 row gathered.  Here:
//   1. all threads list the marked (neighbour, slot) pairs of the point with the codes the join kept for them (join_bounds.hpp);
//   2. the ids of the few hundred with the least codes are gathered and pass a hash set (seeded with the row; drops repeats): what is
//      new goes to the list of candidates;
//   3. the codes say how far the row will reach at most: K of its entries and candidates lie below (join_bounds.hpp).  Where that is
//      beyond the codes taken so far, more of them go through 2 (this is rare);
//   4. the candidates whose bound is not above the reach get the exact distance, the four wavefronts sharing them, at most 256 at a
//      time and nearer bounds first (mostly that is all of them), and
//   5. the row and the new distances, as (distance, index) keys in LDS, are merged by counting: a new key's slot is the number of
//      keys of the row below it (binary search) and of new ones (all of them compared), an old key moves up by the new ones
//      below it.
// A bound is below the exact distance of its pair, the reach is never below the row's final last slot: a dropped
// candidate could not have been in the final row, so the result is the one of any other order.
// (Measured at 70,000 x 784, K = 90: 2,725 marks of 1,466 distinct points, 97 exact distances per point against 140 by rounds without the
// reach and 85 entries that change; 12.6 -> 4.8 ms = 4.6 TB/s of rows.  Of the first form's 188 k cycles per point 50 k were the exact
// distances, 48 k the merge of four rows by insertions, 29 k the set of all marks.  Where marks are many and points few (122,376
// x 4 in 64 clusters, K = 84) the exploration takes a seventh.)
// LDS (ints): set[set_size] | marked[cap], later 4 tiles | ids of the candidates [most] | their codes [most / 2] | srow[K] |
// xrow[dpad] | keys: row [K], merged row [K], new [256] | ids of the new ones [256].
constexpr int kWgChunk = 32;
constexpr int kWgTile = 64 * (kWgChunk + 4);
constexpr int kWgMinCap = 1024;             // the kernel is not used when fewer marks than this would fit
constexpr int kWgMaxCap = 6656;             // marks per point
constexpr int kWgMost = 1536;               // candidates per point
constexpr int kWgMaxSteps = kWgMost / 256;  // of them per thread
constexpr int kWgLeast = 512;               // the kernel is not used when the set has room for fewer
constexpr int kWgGather = 12;               // marks of a thread whose ids are requested together
constexpr int kWgNew = 256;                 // exact distances of a round
static_assert(32 * (2 * kWgChunk + 4) <= kWgTile, "32 rows of twice the dimensions fit the tile");
struct WgSizes { int cap, most, set_size; };

// Candidates c[] (none where negative) into the set, four probes in flight: which of them are new.
__device__ __forceinline__ void set_insert4(int* table, int mask, const int (&c)[4], bool (&fresh)[4])
{
    uint32_t h[4];
    int old[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        h[u] = hash_id(c[u]) & (uint32_t)mask;
        old[u] = c[u] >= 0 ? atomicCAS(&table[h[u]], kEmpty, c[u]) : 0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        fresh[u] = false;
        if (c[u] < 0) continue;
        for (int i = 0; i <= mask; ++i) {
            if (old[u] == kEmpty) { fresh[u] = true; break; }
            if (old[u] == c[u] || old[u] == -c[u] - 1) break;
            h[u] = (h[u] + 1) & (uint32_t)mask;
            old[u] = atomicCAS(&table[h[u]], kEmpty, c[u]);
        }
    }
}

template <int SL>
__global__ __launch_bounds__(256, 3) void k_explore_merge_wg(const float* __restrict__ points, int N, int D, int K,
                                                          const int* __restrict__ old_idx, int* __restrict__ knn_idx,
                                                          float* __restrict__ knn_dist, WgSizes sz, int dpad,
                                                          const uint32_t* __restrict__ pass, JoinBounds jb,
                                                          const int* __restrict__ list, int n_in,
                                                          int* __restrict__ todo_out, int* __restrict__ n_out,
                                                          unsigned long long* __restrict__ stat)
{
    extern __shared__ __align__(16) int lds_w[];
    __shared__ int wave_tot[4], count_s[2][4];
    __shared__ int n_cand_s, n_new_s;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // (the list of points a launch before this one left over is in the order in which that launch came to them)
    const int slot = die_local_place(blockIdx.x, gridDim.x);
    if (slot >= n_in) return;
    const int p = list[slot];
    const int MW = (K + 31) >> 5, KP = MW * 32, kq = (K + 3) & ~3;
    int* table = lds_w;
    uint32_t* marked = reinterpret_cast<uint32_t*>(table + sz.set_size);
    int* tiles = lds_w;                                           // (in the place of the set and the marks)
    int* cand = lds_w + max(sz.set_size + sz.cap, 4 * kWgTile);
    uint16_t* cand_code = reinterpret_cast<uint16_t*>(cand + sz.most);
    int* srow = cand + sz.most + sz.most / 2;
    float* xrow = reinterpret_cast<float*>(srow + kq);
    double* row_key = reinterpret_cast<double*>(xrow + dpad);     // the row, sorted
    double* out_key = row_key + kq;
    double* new_key = out_key + kq;
    int* new_id = reinterpret_cast<int*>(new_key + kWgNew);
    const bool vec_ok = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);

    // The mark words of the point (K MW of them in one piece) are dealt out to the threads; they are requested together with the
    // entries of the snapshot they belong to and with the point's row and coordinates (none of these addresses depends on another's data).
    const int words = K * MW, per_mw = 65536 / MW + 1;            // (word / MW, exact below 2048)
    uint32_t pw[8];                                               // K MW <= 2048
    int pq[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int t = (int)threadIdx.x + 256 * j;
        pw[j] = t < words ? pass[(size_t)p * words + t] : 0u;
        pq[j] = t < words ? old_idx[(size_t)p * K + ((t * per_mw) >> 16)] : -1;
    }
    KnnRow<SL> row;
    row.load(knn_idx + (size_t)p * K, knn_dist + (size_t)p * K, K);
    const float* xp = points + (size_t)p * D;
    for (int d = threadIdx.x; d < dpad; d += 256) xrow[d] = d < D ? xp[d] : 0.0f;
    for (int i = threadIdx.x; i < sz.set_size; i += 256) table[i] = kEmpty;
    int* hist = new_id;                                           // marks by the upper 8 bits of their codes
    hist[threadIdx.x] = 0;

    // ---- 1. the marked pairs of the point
    int mine = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        if (!(pq[j] >= 0 && pq[j] < N)) pw[j] = 0u;               // (the join writes nothing for such entries)
        mine += __popc(pw[j]);
    }
    const int in_wave = wave_excl_scan_i(mine);
    if (lane == 63) wave_tot[wave] = in_wave + mine;
    if (threadIdx.x == 0) {
        n_cand_s = 0;
        n_new_s = 0;
    }
    __syncthreads();
    int at = in_wave, n_marked = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        if (w < wave) at += wave_tot[w];
        n_marked += wave_tot[w];
    }
    if (n_marked == 0) return;
    if (n_marked > sz.cap) {
        if (threadIdx.x == 0) todo_out[atomicAdd(n_out, 1)] = p;
        return;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int t = (int)threadIdx.x + 256 * j;
        if (256 * j >= words) break;
        const int k = (t * per_mw) >> 16, w = t - k * MW;
        if (pw[j]) srow[k] = pq[j];                               // (the same value for every word of the entry)
        uint32_t m = pw[j];
        while (m) {
            const int b = __ffs(m) - 1;
            m &= m - 1;
            marked[at++] = (uint32_t)((32 * w + b) << 8) | (uint32_t)k;
        }
    }
    const int mask = sz.set_size - 1;
    if (wave == 3) {                                              // seeds: the point, and ids that are in the row already
        if (lane == 0) set_insert(table, mask, p, true);
#pragma unroll
        for (int s = 0; s < SL; ++s) {
            if (row.idx[s] >= 0) set_insert(table, mask, row.idx[s], true);
            if (lane + 64 * s < K) row_key[lane + 64 * s] = pair_key(row.dist[s], row.idx[s]);
        }
    }
    __syncthreads();
    const uint16_t* __restrict__ codes_p = jb.codes ? jb.codes + (size_t)p * K * KP : nullptr;
    if (codes_p) {
        for (int i0 = threadIdx.x; i0 < n_marked; i0 += kWgGather * 256) {
            uint32_t e[kWgGather], code[kWgGather];
#pragma unroll
            for (int u = 0; u < kWgGather; ++u) {
                e[u] = i0 + 256 * u < n_marked ? marked[i0 + 256 * u] : 0u;
                code[u] = i0 + 256 * u < n_marked ? codes_p[(e[u] & 255u) * KP + (e[u] >> 8)] : 0u;
            }
#pragma unroll
            for (int u = 0; u < kWgGather; ++u) {
                if (i0 + 256 * u < n_marked) {
                    marked[i0 + 256 * u] = e[u] | code[u] << 16;
                    atomicAdd(&hist[code[u] >> 8], 1);
                }
            }
        }
        __syncthreads();
    }

    const CodeReader codes(jb, p);
    float tau = row.tau;                                          // the last slot, as far as it is known
    int rc[SL];
#pragma unroll
    for (int s = 0; s < SL; ++s) rc[s] = codes.code_of(row.dist[s]);
    int lb16[kWgMaxSteps];                                        // the codes of this thread's candidates: threadIdx.x + 256 u
    int it = 0, n_cand = 0;
    auto count_upto = [&](int from, int upto) {                   // candidates of the workgroup with from < code <= upto
        int n = 0;
#pragma unroll
        for (int u = 0; u < kWgMaxSteps; ++u) {
            if (256 * u >= n_cand) break;
            n += __popcll(ballot64(lb16[u] > from && lb16[u] <= upto));
        }
        ++it;
        if (lane == 0) count_s[it & 1][wave] = n;
        __syncthreads();
        return count_s[it & 1][0] + count_s[it & 1][1] + count_s[it & 1][2] + count_s[it & 1][3];
    };
    int cut = -1;                                                 // marks with codes up to here have become candidates
    for (int want = 6 * K;; want *= 2) {
        // the codes that take at least `want` marks, in steps of 256
        const int from = cut;
        cut = kCodeTop;
        if (codes_p && n_marked > want) {
            int run = 0, bins = 0;
            for (int b0 = 0; b0 < 256; b0 += 64) {
                const int h = hist[b0 + lane];
                const uint64_t below = ballot64(run + wave_excl_scan_i(h) + h < want);     // (a prefix of the bins)
                bins += __popcll(below);
                if (below != ~0ull) break;
                run += wave_sum_i(h);
            }
            cut = max(from, 256 * bins + 255);
        }

        // ---- 2. the distinct ones
        for (int i0 = threadIdx.x; i0 < n_marked; i0 += kWgGather * 256) {
            int c[kWgGather], code[kWgGather];
#pragma unroll
            for (int u = 0; u < kWgGather; ++u) {
                c[u] = -1;
                code[u] = 0;
                if (i0 + 256 * u < n_marked) {
                    const uint32_t e = marked[i0 + 256 * u];
                    code[u] = (int)(e >> 16);
                    if (code[u] > from && code[u] <= cut) c[u] = old_idx[(size_t)srow[e & 255u] * K + ((e >> 8) & 255u)];
                }
                if (c[u] >= N) c[u] = -1;
            }
            for (int g = 0; g < kWgGather; g += 4) {
                if (i0 - (int)threadIdx.x + 256 * g >= n_marked) break;
                if (*reinterpret_cast<volatile int*>(&n_cand_s) > sz.most) break;
                int c4[4], code4[4];
                bool fresh[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    c4[u] = g == 0 ? c[u] : (g == 4 ? c[u + 4] : c[u + 8]);
                    code4[u] = g == 0 ? code[u] : (g == 4 ? code[u + 4] : code[u + 8]);
                }
                set_insert4(table, mask, c4, fresh);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint64_t fm = ballot64(fresh[u]);
                    if (fm == 0) continue;
                    int first = 0;
                    if (lane == 0) first = atomicAdd(&n_cand_s, __popcll(fm));
                    first = __builtin_amdgcn_readfirstlane(first) + mask_prefix(fm);
                    if (fresh[u] && first < sz.most) {
                        cand[first] = c4[u];
                        cand_code[first] = (uint16_t)code4[u];
                    }
                }
            }
        }
        __syncthreads();
        n_cand = n_cand_s;
        if (n_cand > sz.most) {                                   // too many that may matter
            if (threadIdx.x == 0) todo_out[atomicAdd(n_out, 1)] = p;
            return;
        }

        // ---- 3. how far the row reaches (every wavefront for itself: no barriers)
        if (codes_p) {
            constexpr int kIn = kWgMost / 64;
            int lo = 1, hi = kCodeTop;
            if (n_cand <= 64 * (kIn / 2)) {
                int cc[kIn / 2];
#pragma unroll
                for (int u = 0; u < kIn / 2; ++u) {
                    const int b = 64 * u + lane < n_cand ? (int)cand_code[64 * u + lane] : 0;
                    cc[u] = b > 0 ? b : kCodeTop;
                }
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    int n = 0;
#pragma unroll
                    for (int u = 0; u < kIn / 2; ++u) {
                        if (64 * u >= n_cand) break;
                        n += __popcll(ballot64(cc[u] <= mid));
                    }
#pragma unroll
                    for (int s = 0; s < SL; ++s) n += __popcll(ballot64(rc[s] <= mid));
                    if (n >= K) hi = mid;
                    else lo = mid + 1;
                }
            } else {
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    int n = 0;
                    for (int t0 = 0; t0 < n_cand; t0 += 64) {
                        const int b = t0 + lane < n_cand ? (int)cand_code[t0 + lane] : 0;
                        n += __popcll(ballot64(b > 0 && b <= mid));
                    }
#pragma unroll
                    for (int s = 0; s < SL; ++s) n += __popcll(ballot64(rc[s] <= mid));
                    if (n >= K) hi = mid;
                    else lo = mid + 1;
                }
            }
            if (lo < kCodeTop) tau = fminf(tau, codes.reach(lo));
        }
        if (cut >= kCodeTop || codes.last_code(tau) <= cut) break;
        __syncthreads();                                          // (n_cand_s has been read)
    }
    if (n_cand == 0) return;
#pragma unroll
    for (int u = 0; u < kWgMaxSteps; ++u) {
        const int i = threadIdx.x + 256 * u;
        lb16[u] = i < n_cand ? (int)cand_code[i] : 0x7fffffff;
    }

    // ---- 4. the exact distances of a round
    float* tile = reinterpret_cast<float*>(tiles + wave * kWgTile);
    const int k = threadIdx.x;                                    // (the slot of the row and the new key this thread places)
    bool changed = false;
    int n_exact = 0;
    while (true) {
        const int last = codes_p ? codes.last_code(tau) : kCodeTop;
        const int n_left = count_upto(-1, last);                  // (a barrier: the set, and the keys of the round before, have been read)
        if (n_left == 0) break;
        int upto = last;
        if (n_left > kWgNew) {
            // the least codes of them (equal codes: any of them)
            int lo = 0;
            while (lo < upto) {
                const int mid = (lo + upto) >> 1;
                if (count_upto(-1, mid) >= kWgNew / 4 * 3) upto = mid;
                else lo = mid + 1;
            }
        }
#pragma unroll
        for (int u = 0; u < kWgMaxSteps; ++u) {
            if (256 * u >= n_cand) break;
            const bool take = lb16[u] <= upto;
            const uint64_t m = ballot64(take);
            if (m == 0) continue;
            int first = 0;
            if (lane == 0) first = atomicAdd(&n_new_s, __popcll(m));
            first = __builtin_amdgcn_readfirstlane(first) + mask_prefix(m);
            if (take && first < kWgNew) {
                new_id[first] = cand[threadIdx.x + 256 * u];
                lb16[u] = 0x7fffffff;
            }
        }
        __syncthreads();
        const int n = min(kWgNew, n_new_s);
        const int share = (n + 3) >> 2, own = min(wave * share, n), n_own = min(share, n - own);      // at most 64
        if (n_own > 0) {
            float d;
            bool finished;
            if (share <= 32) finished = exact_distances<2 * kWgChunk, 32, true, kChainGroup>(tile, xrow, new_id + own, n_own, points, D, vec_ok, tau, d);
            else finished = exact_distances<kWgChunk, 64, true, kChainGroup>(tile, xrow, new_id + own, n_own, points, D, vec_ok, tau, d);
            // (what cannot enter: a key above all others)
            if (lane < n_own) new_key[own + lane] = finished && d < INFINITY ? pair_key(d, new_id[own + lane]) : INFINITY;
            n_exact += n_own;
        }
        if (threadIdx.x == 0 && (n & 1)) new_key[n] = INFINITY;   // (read in twos)
        __syncthreads();
        if (threadIdx.x == 0) n_new_s = 0;
        // ---- 5. the row and the new keys (pairs are distinct, but for empty slots of the row)
        const double mine_old = k < K ? row_key[k] : INFINITY, mine_new = k < n ? new_key[k] : INFINITY;
        int rank_old = k, rank_new = 0;
        for (int step = 256; step > 0; step >>= 1)
            if (rank_new + step <= K && row_key[rank_new + step - 1] < mine_new) rank_new += step;
        for (int i = 0; i < n; i += 2) {
            const double2 v = *reinterpret_cast<const double2*>(new_key + i);
            rank_old += v.x < mine_old ? 1 : 0;
            rank_old += v.y < mine_old ? 1 : 0;
            rank_new += v.x < mine_new ? 1 : 0;
            rank_new += v.y < mine_new ? 1 : 0;
        }
        const bool enters = k < n && mine_new < INFINITY && rank_new < K;
        if (k < K && rank_old < K) out_key[rank_old] = mine_old;
        if (enters) out_key[rank_new] = mine_new;
        const uint64_t em = ballot64(enters);
        ++it;
        if (lane == 0) count_s[it & 1][wave] = em != 0;
        __syncthreads();
        if (count_s[it & 1][0] | count_s[it & 1][1] | count_s[it & 1][2] | count_s[it & 1][3]) {
            changed = true;
            double* t = row_key;
            row_key = out_key;
            out_key = t;
            tau = fminf(tau, pair_dist(row_key[K - 1]));
        }
    }
    count_exact(stat, n_exact);
    if (changed && k < K) {
        const double v = row_key[k];
        knn_idx[(size_t)p * K + k] = __double2loint(v);
        knn_dist[(size_t)p * K + k] = pair_dist(v);
    }
}

// Sizes of the workgroup-per-point merge, with the LDS of a compute unit shared by three workgroups where they have room for the marks a
// point can have, else by two; no marks (cap) at all where it does not fit.
int merge_wg_ints(const WgSizes& sz, int dpad, int K)
{
    return (std::max(sz.set_size + sz.cap, 4 * kWgTile) + sz.most + sz.most / 2 + dpad + 5 * ((K + 3) & ~3) + 3 * kWgNew + 3) / 4 * 4;
}

WgSizes merge_wg_sizes(int dpad, int K)
{
    // three workgroups per compute unit where that leaves room for kWgMaxCap marks, else two
    for (int share = 3; share >= 2; --share) {
        const int budget = (160 * 1024 / share - 1024) / 4;
        for (int set = 2048; set >= 1024; set >>= 1) {
            WgSizes sz;
            sz.set_size = set;
            sz.most = std::min(kWgMost, (set / 8 * 7 - K - 1) & ~7);
            if (sz.most < kWgLeast) continue;
            sz.cap = std::min({budget - merge_wg_ints({0, sz.most, set}, dpad, K) + std::max(0, 4 * kWgTile - set), K * K + 3, kWgMaxCap}) & ~3;
            const int enough = share == 3 ? std::min((K * K + 3) & ~3, kWgMaxCap) : kWgMinCap;
            if (sz.cap >= enough && sz.cap >= kWgMinCap && merge_wg_ints(sz, dpad, K) <= budget) return sz;
        }
    }
    return {0, 0, 0};
}

template <int SL>
int launch_merge_wg(const float* points, int N, int D, int K, const int* old_idx, int* knn_idx, float* knn_dist,
                    const WgSizes& sz, int dpad, const uint32_t* pass, const JoinBounds& bounds, const int* list, int n_in,
                    int* todo_out, int* n_out, unsigned long long* stat, hipStream_t stream)
{
    const size_t lds = (size_t)merge_wg_ints(sz, dpad, K) * sizeof(int);
    RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_explore_merge_wg<SL>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    for (int off = 0; off < n_in; off += kMostGroups) {       // (as many points as a launch has threads for)
        const int n = std::min(n_in - off, kMostGroups);
        hipLaunchKernelGGL((k_explore_merge_wg<SL>), dim3(grid_for_dies((size_t)n)), dim3(256), lds, stream, points, N, D, K, old_idx,
                           knn_idx, knn_dist, sz, dpad, pass, bounds, list + off, n, todo_out, n_out, stat);
    }
    RSFK_HIP(hipGetLastError());
    return 0;
}

int next_pow2(int v)
{
    int p = 1;
    while (p < v) p <<= 1;
    return p;
}

template <int SL, int WAVES>
int launch_merge(const float* points, int N, int D, int K, const int* old_idx, int* knn_idx, float* knn_dist, int table,
                 int wave_ints, int dpad, bool direct, const uint32_t* pass, const JoinBounds& bounds, const int* todo_in, int n_in,
                 int* todo_out, int share, int* n_out, unsigned long long* stat, const int* order, hipStream_t stream)
{
    const size_t lds = (size_t)WAVES * (size_t)wave_ints * sizeof(int);
    const int n_work = todo_in ? n_in : N;
    dim3 grid(grid_for_dies(((size_t)n_work + WAVES - 1) / WAVES)), block(64 * WAVES);
    auto* kernel = !direct                                         ? k_explore_merge<SL, WAVES, kFormTile>
                   : !merge_quads(N, D, K, bounds.codes != nullptr) ? k_explore_merge<SL, WAVES, kFormOwn>
                   : bounds.codes                                  ? k_explore_merge<SL, WAVES, kFormDirectCoded>
                                                                   : k_explore_merge<SL, WAVES, kFormDirect>;
    RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, points, N, D, K, old_idx, knn_idx, knn_dist, table, wave_ints, dpad, pass,
                       bounds, todo_in, n_in, todo_out, share, n_out, stat, order);
    RSFK_HIP(hipGetLastError());
    return 0;
}

// ints of LDS a wavefront of the merge kernel needs for a set of `table` entries: tile | point | set | row | list of
// marks | with_bounds: a bound per place of the set
int merge_wave_ints(int table, int dpad, int K, bool with_bounds, int tile)
{
    const int lists = table + K + table / 4 * 3 + (with_bounds ? table : 0);
    const int ranks = tile > 0 ? 0 : merge_rank_at(table, K, with_bounds) + rank_words(row_slots(K));
    return (tile + dpad + std::max(lists, ranks) + 3) / 4 * 4;
}
int merge_wave_ints(int table, int dpad, int K, bool with_bounds = false)
{
    return merge_wave_ints(table, dpad, K, with_bounds, merge_tile_ints(dpad, merge_direct_max()));
}

int dispatch_merge(int sl, int waves, const float* points, int N, int D, int K, const int* old_idx, int* knn_idx,
                   float* knn_dist, int table, int dpad, const uint32_t* pass, const JoinBounds& bounds, const int* todo_in,
                   int n_in, int* todo_out, int share, int* n_out, unsigned long long* stat, const int* order, hipStream_t stream)
{
    const bool coded = bounds.codes != nullptr, direct = merge_direct(D, dpad, coded);
    const int wi = merge_wave_ints(table, dpad, K, coded, direct ? 0 : kMergeTile);
#define RSFK_MERGE_CASE(SLV, WV)                                                                                        \
    if (sl == SLV && waves == WV)                                                                                       \
        return launch_merge<SLV, WV>(points, N, D, K, old_idx, knn_idx, knn_dist, table, wi, dpad, direct, pass, bounds, \
                                     todo_in, n_in, todo_out, share, n_out, stat, order, stream);
    RSFK_MERGE_CASE(1, 4) RSFK_MERGE_CASE(1, 2) RSFK_MERGE_CASE(1, 1)
    RSFK_MERGE_CASE(2, 4) RSFK_MERGE_CASE(2, 2) RSFK_MERGE_CASE(2, 1)
    RSFK_MERGE_CASE(4, 4) RSFK_MERGE_CASE(4, 2) RSFK_MERGE_CASE(4, 1)
#undef RSFK_MERGE_CASE
    RSFK_CHECK(false, "exploration: no merge kernel for this configuration");
}

// The shares of a list to one list (a workgroup each).
__global__ __launch_bounds__(256) void k_todo_join(const int* __restrict__ lists, int share, const int* __restrict__ numbers, int* __restrict__ out)
{
    const int s = blockIdx.x, lane = threadIdx.x & 63;
    const int mine = lane < kTodoShares ? numbers[32 * lane] : 0, n = read_lane_i(mine, s);
    const int at = wave_sum_i(lane < s ? mine : 0);
    for (int i = threadIdx.x; i < n; i += 256) out[at + i] = lists[(size_t)s * (size_t)share + i];
}

template <int SL, int WAVES>
int launch_one(const float* points, const Bf16Copy& b, int N, int D, int K, const int* old_idx, int* knn_idx,
               float* knn_dist, int table, int wave_ints, int dpad, int rows_per_group, const int* todo, int n_todo,
               unsigned long long* stat, hipStream_t stream)
{
    const size_t lds = (size_t)WAVES * (size_t)wave_ints * sizeof(int);
    RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_explore<SL, WAVES>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int n_work = todo ? n_todo : N;
    for (int first = 0; first < n_work; first += std::min(kMostRows, n_work - first)) {
        dim3 grid((unsigned)((std::min(kMostRows, n_work - first) + WAVES - 1) / WAVES)), block(64 * WAVES);
        hipLaunchKernelGGL((k_explore<SL, WAVES>), grid, block, lds, stream, points, b, N, D, K, old_idx, knn_idx, knn_dist,
                           table, wave_ints, dpad, rows_per_group, todo, first, n_todo, stat);
    }
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// Does the join keep the lower bounds of the pairs it marks (N K KP 2-byte words)?  Yes for the rows that go to the
// workgroup-per-point merge (below), and for rows of more than 128 dimensions while the array stays below 4 GB: the
// wavefront-per-point merge then takes the candidates of a point nearer bounds first (their rows are long, and every
// candidate that a tighter last slot turns away is a row not read).  Up to 128 dimensions they cost more than they give, without -> with:
// 1M x 100, 50 trees, join 3.44 -> 4.81 ms and merge 2.74 -> 3.24, in 64 clusters 3.03 -> 4.50 and 2.62 -> 3.29; 1M x 128 3.53 -> 4.92 and
// 2.79 -> 3.39; 300,000 x 64, K = 48, 12 trees 1.12 -> 2.35 and 1.46 -> 2.03, x 128, K = 60 2.27 -> 3.92 and 8.46 -> 7.70.
// RSFK_MERGE_ORDER=0 switches the second case off.
bool explore_join_keeps_bounds(int N, int D, int K)
{
    if (explore_merge_uses_bounds(D, K)) return true;
    static const bool on = [] {
        const char* e = std::getenv("RSFK_MERGE_ORDER");
        return !(e && e[0] == '0');
    }();
    const size_t KP = (size_t)((K + 31) & ~31);
    return on && D > 128 && K <= 64 && (size_t)N * (size_t)K * KP * 2 <= ((size_t)4 << 30);
}

bool explore_merge_uses_bounds(int D, int K)
{
    const int dpad = bf16_valid(D);
    const int lds_ints = 150 * 1024 / 4;
    const int want = std::max(next_pow2(K * K + K + 2), next_pow2(4 * K + 66));
    int big_waves = 4;
    while (big_waves > 1 && merge_wave_ints(want, dpad, K) > lds_ints / big_waves) big_waves >>= 1;
    return big_waves < 4 && merge_wg_sizes(dpad, K).cap > 0;
}

// Rows short enough for the LDS of the merge kernels: the exploration then takes its candidates from the join, and
// the general kernel (the only user of the bfloat16 copy) only sees what the merge kernels hand back.
bool explore_merge_fits(int D, int K)
{
    const int small_table = std::min(4096, std::max(256, next_pow2(16 * K)));
    return K <= kMaxKJoin && 4 * merge_wave_ints(small_table, bf16_valid(D), K) <= 150 * 1024 / 4;
}

// One exploration pass.  old_idx is scratch of N*K ints (receives the snapshot).
// bf may be null (or hold null rows): every candidate then gets the exact distance.
// ws may be null; with a workspace and the copy for the join (jc)
// the candidates come from the join over the reversed graph (explore_join.hip), which needs rows sorted by
// distance.
int launch_explore(const float* points, const Bf16Copy* bf, const JoinCopy* jc, int N, int D, int K, int* knn_idx,
                   float* knn_dist, int* old_idx, ExploreWorkspace* ws, hipStream_t stream, bool rows_sorted,
                   unsigned long long* stat, const int* order, bool one_tree)
{
    if (N <= 0) return 0;
    RSFK_CHECK(K >= 1 && K <= kMaxK, "exploration: K must be in 1..1024");
    const int dpad = bf16_valid(D);
    const int small_table = std::min(4096, std::max(256, next_pow2(16 * K)));
    // (rows too long for the LDS of the merge kernel: every point enumerates its own candidates)
    const bool join = ws != nullptr && jc != nullptr && jc->rows != nullptr && explore_merge_fits(D, K);
    // (rows_sorted: the caller knows that every row is in order, e.g. after the bucket step of a forest)
    if (join && !rows_sorted && launch_sort_rows(knn_idx, knn_dist, N, K, stream)) return 1;
    if (!join) RSFK_HIP(hipMemcpyAsync(old_idx, knn_idx, sizeof(int) * (size_t)N * (size_t)K, hipMemcpyDeviceToDevice, stream));
    const int fixed = 64 * kPitch + dpad + kQueue2 + K;                 // ints per wavefront besides the set
    const int lds_ints = 150 * 1024 / 4;                                // usable LDS per workgroup
    // The set must hold the seeds (K+1) and all candidates of a group of neighbours with room to
    // spare.  Prefer 4 wavefronts per workgroup; shrink the workgroup, then the group of
    // neighbours, when K is large.
    // (the kernel walks the set 64 entries at a time: it must never be smaller than 64)
    const int floor_table = next_pow2(4 * K + 66);
    const int want = std::max(next_pow2(K * K + K + 2), floor_table);
    RSFK_CHECK(fixed + floor_table <= lds_ints, "exploration: D or K too large for the LDS budget");
    int waves = 4;
    int table = want;
    while (waves > 1 && fixed + table > lds_ints / waves) waves >>= 1;
    while (table > floor_table && fixed + table > lds_ints / waves) table >>= 1;
    int rows_per_group = K;
    if (table < want) rows_per_group = std::max(1, (table * 3 / 4 - K - 1) / K);
    RSFK_CHECK(table >= 64 && (table & (table - 1)) == 0 && rows_per_group >= 1, "exploration: bad set size");
    const int wave_ints = (fixed + table + 3) / 4 * 4;
    Bf16Copy b;
    if (bf) b = *bf;
    const int sl = row_slots(K);
    const int* todo = nullptr;
    int n_todo = 0;
    if (join) {
        // Marks from the join, then the merge kernel with a small set (little LDS, many wavefronts per CU).
        // The points it cannot take come back in a list and get a second launch with the largest set that
        // fits; what is left after that goes to the general kernel below.
        if (launch_explore_join(ws, *jc, N, D, K, knn_idx, old_idx, knn_dist, stream, order)) return 1;
        const uint32_t* pass = explore_ws_pass(ws);
        int* listA = explore_ws_todo(ws, 0);
        int* listB = explore_ws_todo(ws, 1);
        int* lists = explore_ws_share_lists(ws);          // what the small set hands back, in shares; listA once they are joined
        int* numbers = explore_ws_shares(ws);
        const int share = todo_share(N);
        int n_back = 0;
        // (the bounds of the join, when it kept them and the set with a bound per place still fits)
        JoinBounds wave_bounds = explore_ws_bounds(ws), no_bounds = wave_bounds;
        no_bounds.codes = nullptr;
        if (4 * merge_wave_ints(small_table, dpad, K, true) > lds_ints) wave_bounds = no_bounds;
        int big_table = want, big_waves = 4;
        while (big_waves > 1 && merge_wave_ints(big_table, dpad, K) > lds_ints / big_waves) big_waves >>= 1;
        // fewer than four wavefronts per workgroup would leave the compute units nearly empty: such sets get one
        // workgroup per point instead.  So do sets of 2048 places and more where the join kept its codes (at least one workgroup of
        // four of them fits a compute unit, but they evaluate every candidate, and that kernel what the codes leave):
        // whole pass with points that have most of their marks, D = 132, K = 40 5.4 -> 4.5 ms, K = 50 14.1 -> 6.0; D = 256, K = 32
        // 9.2 -> 4.9, K = 60 28.6 -> 8.0; D = 960, K = 60 36.5 -> 5.9.  Not with K = 32 while two workgroups fit (120,000 points after two trees, by
        // wavefronts -> by workgroups: D = 192 3.21 -> 3.55 ms, 224 3.56 -> 3.82, 256 6.38 -> 3.89, in clusters after four 192 2.93 -> 3.33, 224 3.29 ->
        // 3.66, 256 5.51 -> 3.79), and not after one tree, when the many marks of a point are the few points of its bucket (D = 132, K = 38 2.36 ->
        // 5.13, D = 192, K = 32 1.75 -> 3.99, K = 60 7.48 -> 8.98, D = 420, K = 60 9.79 -> 10.16).
        const WgSizes wg = merge_wg_sizes(dpad, K);
        const bool by_codes = explore_ws_bounds(ws).codes != nullptr && big_table >= 2048 && !one_tree && wg.cap > 0 &&
                              (K > 32 || merge_wave_ints(big_table, dpad, K) > 80 * 1024 / 16);
        const bool per_wg = big_waves < 4 || by_codes;
        if (!per_wg)
            while (big_table > small_table && merge_wave_ints(big_table, dpad, K) > lds_ints / big_waves) big_table >>= 1;
        const bool second = per_wg ? wg.cap > 0 : big_table > small_table;
        auto merge_wg = [&](const int* list, int n) {
            const JoinBounds& bounds = explore_ws_bounds(ws);
            if (sl == 1)
                return launch_merge_wg<1>(points, N, D, K, old_idx, knn_idx, knn_dist, wg, dpad, pass, bounds, list, n, listB,
                                          listB + N, stat, stream);
            if (sl == 2)
                return launch_merge_wg<2>(points, N, D, K, old_idx, knn_idx, knn_dist, wg, dpad, pass, bounds, list, n, listB,
                                          listB + N, stat, stream);
            return launch_merge_wg<4>(points, N, D, K, old_idx, knn_idx, knn_dist, wg, dpad, pass, bounds, list, n, listB,
                                      listB + N, stat, stream);
        };
        // Where the workgroup-per-point kernel may follow, the small set is first tried on a sample (the first points of
        // the order they are taken in): when it has to hand most of them back -- rows of many neighbours that are far
        // from done have thousands of marks each -- the launch over all points would only find that out for every
        // one of them (70,000 x 784, K = 90, 10 trees: all of them, 0.9 ms of a 25 ms pass).
        constexpr int kSample = 2048;                      // (a multiple of kTodoShares: no share holds more than its part of N)
        int first = 0;                                    // points the small set has been tried on
        bool rest_per_wg = false;
        if (second && per_wg && order != nullptr && N > 2 * kSample) {
            if (dispatch_merge(sl, 4, points, N, D, K, old_idx, knn_idx, knn_dist, small_table, dpad, pass, wave_bounds, order,
                               kSample, lists, share, numbers, stat, nullptr, stream))
                return 1;
            if (fetch_total(numbers, kTodoShares, 32, &n_back, stream)) return 1;
            first = kSample;
            rest_per_wg = n_back > kSample / 2;
        }
        if (rest_per_wg) {
            // everything but the sample straight to the workgroup-per-point kernel (its list: the rest of the order)
            if (merge_wg(order + first, N - first)) return 1;
        } else if (dispatch_merge(sl, 4, points, N, D, K, old_idx, knn_idx, knn_dist, small_table, dpad, pass, wave_bounds,
                                  first > 0 ? order + first : nullptr, first > 0 ? N - first : 0, lists, share, numbers, stat,
                                  first > 0 ? nullptr : order, stream)) {
            return 1;
        }
        if (fetch_total(numbers, kTodoShares, 32, &n_back, stream)) return 1;
        // (20,000 x 32 in 64 clusters, K = 32: 11,193 points come back, one counter took 0.10 of the launch's 0.136 ms)
        if (n_back > 0) hipLaunchKernelGGL(k_todo_join, dim3(kTodoShares), dim3(256), 0, stream, lists, share, numbers, listA);
        n_todo = n_back;                                 // what the small set handed back (of the sample, or of all points)
        todo = listA;
        if (n_todo == 0 && !rest_per_wg) return 0;
        if (second) {
            int rc = 0;
            if (n_todo == 0)
                rc = 0;
            else if (!per_wg)
                rc = dispatch_merge(sl, big_waves, points, N, D, K, old_idx, knn_idx, knn_dist, big_table, dpad, pass,
                                    no_bounds, listA, n_todo, listB, 0, listB + N, stat, nullptr, stream);
            else
                rc = merge_wg(listA, n_todo);
            if (rc)
                return 1;
            if (fetch_words(listB + N, 1, &n_back, stream)) return 1;
            n_todo = n_back;
            if (n_todo == 0) return 0;
            todo = listB;
        }
    }
#define RSFK_EXPLORE_CASE(SLV, WV)                                                                                      \
    if (sl == SLV && waves == WV)                                                                                       \
        return launch_one<SLV, WV>(points, b, N, D, K, old_idx, knn_idx, knn_dist, table, wave_ints, dpad,              \
                                   rows_per_group, todo, n_todo, stat, stream);
    RSFK_EXPLORE_CASE(1, 4) RSFK_EXPLORE_CASE(1, 2) RSFK_EXPLORE_CASE(1, 1)
    RSFK_EXPLORE_CASE(2, 4) RSFK_EXPLORE_CASE(2, 2) RSFK_EXPLORE_CASE(2, 1)
    RSFK_EXPLORE_CASE(4, 4) RSFK_EXPLORE_CASE(4, 2) RSFK_EXPLORE_CASE(4, 1)
    RSFK_EXPLORE_CASE(8, 4) RSFK_EXPLORE_CASE(8, 2) RSFK_EXPLORE_CASE(8, 1)
    RSFK_EXPLORE_CASE(16, 4) RSFK_EXPLORE_CASE(16, 2) RSFK_EXPLORE_CASE(16, 1)
#undef RSFK_EXPLORE_CASE
    RSFK_CHECK(false, "exploration: no kernel for this configuration");
}

}  // namespace rsfk
