// Query-set search: query points are routed through a tree built on the base points and every base point
// of the leaf a query reaches is offered to the query's K-NN row.  Replaces the per-tree part of
// RSFK::knn_gpu_rsfk_forest_ann_tree (src/rsfk.cu:262-441): the level loop that moves the queries down
// (build_tree_check_active_points / build_tree_check_points_side / build_tree_update_parents_ann, one launch and
// one device synchronisation each per level) and compute_knn_from_buckets_perwarp_coalesced_ann
// (src/kernels/build_tree_update_parents_ann.cu:239-517).
//
// The tree builder records an index of each tree on request (TreeRec: the drawn pair and the children of every
// node, the segment of every bucket), so a query descends the whole tree in one kernel: a half wavefront per
// query recomputes the hyperplane of a node from its pair and takes the side test with the arithmetic of the
// builder (32 lane-strided partial sums + xor butterfly: build_tree_check_points_side.cu:131-149,
// create_node.cu:122-135); a node with one child (empty side, or the min-size merge) needs no test and is not in
// the index.
//
// The queries are then grouped by the bucket they reached (a count per bucket taken while routing, a scan, a fill)
// and a workgroup works on one bucket and up to 16 of its queries: the rows of the bucket pass through LDS once per
// workgroup instead of once per query, every lane runs the sequential chain of "its" bucket member against four
// queries whose coordinates are wavefront-uniform, and the candidates are merged into the queries' rows.  Trees after which
// few pairs still enter a row are searched by the kernel of ann_screen.hip instead, which bounds the pairs first.
//
// That is a chain of six launches per tree, which a small set of queries cannot fill; its trees go together instead
// (launch_ann_forest): the queries are routed through all trees in one launch, and one workgroup per query works on the
// buckets the query reached in all of them.
#include "forest.hpp"
#include "ann.hpp"
#include "exact_batch.hpp"
#include <algorithm>
#include <cstdlib>

namespace rsfk {

namespace {

constexpr int kQB = kAnnDirect;       // queries per workgroup
constexpr int kLeafGrid = 4096;       // workgroups of k_ann_leaf
constexpr int kAnnScreenDims = 4096;  // the bounds of the screened form are useless long before
constexpr int kQW = 4;                // queries a wavefront works on together
constexpr int kCG = 128;              // bucket members per pass: two per lane
constexpr int kCH = 32;               // dimensions per staging step
constexpr int kTP = kCH + 4;          // tile pitch: odd number of 16-byte units
constexpr int kPieces = kCH / 4;      // 16-byte pieces of a row per staging step = lanes per row
constexpr int kRowsPer = 256 / kPieces;   // rows per load instruction of the workgroup
constexpr int kLoads = kCG / kRowsPer;    // load instructions per staging step

__global__ __launch_bounds__(256) void k_zero_ints(int* __restrict__ p, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Hyperplane of every two-child node of the index, one wavefront per record: row r of `planes` (pitch floats) is
// [offset, 0, 0, 0 | normal, zero padded to a multiple of 4].  Normal and offset are the values the builder works with
// (create_node.cu:122-135: n = x1 - x2, offset = sum n_d (x1_d + x2_d) / 2 as 32 lane-strided partial sums + xor butterfly).
// blockIdx.y: the tree; the records and the rows of a tree begin rec_cap after those of the tree before it.
// low (null: none): the rows the queries are routed by first, low_pitch floats each: {-b~ (NaN: never certain), 0, children | n~}
// (SideBound, ann.hpp; mu, scale: of the copy of the queries).  A bucket has children -1.
__global__ __launch_bounds__(256) void k_planes(const float* __restrict__ points, int D, const TreeRec* __restrict__ recs,
                                                const int* __restrict__ n_rec_p, int rec_cap, float* __restrict__ planes,
                                                int pitch, float* __restrict__ low, int low_pitch, const float* __restrict__ mu, const float* __restrict__ scale)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6), j = blockIdx.y;
    if (r >= min(n_rec_p[kTreeStatPitch * j], rec_cap)) return;
    const size_t at = (size_t)j * (size_t)rec_cap + (size_t)r;
    const TreeRec rec = recs[at];
    float* low_row = low ? low + at * (size_t)low_pitch : nullptr;
    if (rec.c0 < 0) {
        if (low && lane == 0) *reinterpret_cast<int4*>(low_row) = make_int4(0, 0, -1, -1);
        return;
    }
    const float* x1 = points + (size_t)rec.a * (size_t)D;
    const float* x2 = points + (size_t)rec.b * (size_t)D;
    float* row = planes + at * (size_t)pitch;
    float s = 0.0f;
    if (lane < 32) {
        for (int d = lane; d < D; d += 32) {
            const float t1 = x1[d], t2 = x2[d];
            const float nd = t1 - t2;
            const float prod = nd * (t1 + t2);
            s = s + prod * 0.5f;
        }
    }
    s = half_butterfly_sum(s);
    if (lane < 4) row[lane] = lane == 0 ? s : 0.0f;
    for (int d = lane; d < pitch - 4; d += 64) row[4 + d] = d < D ? x1[d] - x2[d] : 0.0f;
    if (!low) return;
    const RoundedPlane pl = rounded_plane(x1, x2, D, __shfl(s, 0, 64), mu, *scale);
    uint16_t* low_n = reinterpret_cast<uint16_t*>(low_row + 4);
    for (int d = lane; d < ((D + 7) & ~7); d += 64) low_n[d] = rounded_value(d < D ? x1[d] - x2[d] : 0.0f, pl);
    if (lane == 0)
        *reinterpret_cast<int4*>(low_row) = make_int4(__float_as_int(pl.sound ? -pl.b : __builtin_nanf("")), 0, rec.c0, rec.c1);
}

// Eight lanes per query.  A lane owns four of the 32 partial sums of the side test (sums 4s..4s+3 of
// build_tree_check_points_side.cu:131-149: sum j takes the dimensions j, j+32, ... in turn) and adds them in the order
// of the xor butterfly; the other three steps of the butterfly run over the eight lanes.  The first 128 dimensions of
// the query stay in registers.  q_rec[q] = record of the bucket reached, q_rank[q] = arrival number of q among the
// queries of that bucket (cnt counts them, at record << cnt_shift).  FOREST: blockIdx.y is the tree, and reached[q T + tree] = {start, size} of
// the bucket is all that is kept.
constexpr int kXR = 4;
template <bool VEC, bool FOREST>
__global__ __launch_bounds__(256) void k_route(const float* __restrict__ planes, int pitch, const float* __restrict__ queries,
                                               int NQ, int D, const TreeRec* __restrict__ recs, int max_steps,
                                               const int* __restrict__ start, int* __restrict__ q_rec, int* __restrict__ q_rank, int* __restrict__ cnt,
                                               int cnt_shift, int2* __restrict__ reached)
{
    if (FOREST) {
        recs += (size_t)blockIdx.y * (size_t)max_steps;         // (max_steps: the records a tree has room for)
        planes += (size_t)blockIdx.y * (size_t)max_steps * (size_t)pitch;
    }
    const int sub = threadIdx.x & 7;
    const int q = (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 3);
    const bool valid = q < NQ;
    const float* x = queries + (size_t)(valid ? q : 0) * (size_t)D;
    const int Dp = pitch - 4;
    float4 xr[kXR];
#pragma unroll
    for (int k = 0; k < kXR; ++k) xr[k] = load_piece(x, 32 * k + 4 * sub, D, VEC);
    int cur = start && valid ? start[q] : 0;             // (where the first levels have been taken already: ann_top.hip)
    bool done = !valid;
    for (int step = 0; step <= max_steps; ++step) {          // a path is never longer than the number of records
        const int at = done ? 0 : cur;
        const TreeRec r = recs[at];
        const float* pl = planes + (size_t)at * (size_t)pitch;   // requested together with the record; unused for a bucket
        const float b = pl[0];
        float4 n4[kXR];
#pragma unroll
        for (int k = 0; k < kXR; ++k) {
            const int d = 32 * k + 4 * sub;
            n4[k] = d < Dp ? *reinterpret_cast<const float4*>(pl + 4 + d) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
        for (int k = 0; k < kXR; ++k) {
            s0 = __builtin_fmaf(n4[k].x, xr[k].x, s0);
            s1 = __builtin_fmaf(n4[k].y, xr[k].y, s1);
            s2 = __builtin_fmaf(n4[k].z, xr[k].z, s2);
            s3 = __builtin_fmaf(n4[k].w, xr[k].w, s3);
        }
        for (int d0 = 32 * kXR; d0 < D; d0 += 64) {            // two steps of the chains per trip
            const int da = d0 + 4 * sub, db = da + 32;
            const float4 na = da < Dp ? *reinterpret_cast<const float4*>(pl + 4 + da) : make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 nb = db < Dp ? *reinterpret_cast<const float4*>(pl + 4 + db) : make_float4(0.f, 0.f, 0.f, 0.f);
            const float4 xa = load_piece(x, da, D, VEC), xb = load_piece(x, db, D, VEC);
            s0 = __builtin_fmaf(na.x, xa.x, s0); s1 = __builtin_fmaf(na.y, xa.y, s1);
            s2 = __builtin_fmaf(na.z, xa.z, s2); s3 = __builtin_fmaf(na.w, xa.w, s3);
            s0 = __builtin_fmaf(nb.x, xb.x, s0); s1 = __builtin_fmaf(nb.y, xb.y, s1);
            s2 = __builtin_fmaf(nb.z, xb.z, s2); s3 = __builtin_fmaf(nb.w, xb.w, s3);
        }
        float t = (s0 + s1) + (s2 + s3);
        t += dpp_f<kDppXor1>(t);
        t += dpp_f<kDppXor2>(t);
        t += dpp_f<kDppHalfMirror>(t);
        if (!done) {
            if (r.c0 < 0) {
                if (FOREST) {
                    if (sub == 0) reached[(size_t)q * gridDim.y + blockIdx.y] = make_int2(r.a, r.b);
                } else if (sub == 0) {
                    q_rec[q] = cur;
                    q_rank[q] = atomicAdd(&cnt[cur << cnt_shift], 1);
                }
                done = true;
            } else {
                cur = t < b ? r.c1 : r.c0;
            }
        }
        if (ballot64(!done) == 0) break;
    }
}

// The same for many queries of up to 128 dimensions, by the rounded hyperplanes of k_planes and the rounded queries of jc, 8 NH dimensions per
// lane and two per instruction (v_dot2_f32_f16); a test that is not certain is taken exactly.
// Bound by the hyperplanes that miss the L2 (4.3 TB/s of them, vector ALUs half busy), hence their two cache lines.  1M queries, a tree
// of 1M x 100: 0.48 ms with bfloat16 hyperplanes, fp32 queries and all levels, 0.27 where ann_top.hip has taken the first seven.  Tried:
// the queries of a subtree on one die (misses 9.4 -> 5.4 million lines, but the queries come in no order then: 0.44).
template <int NH>
__global__ __launch_bounds__(256) void k_route_low(const float* __restrict__ planes, int pitch, const float* __restrict__ low, int low_pitch,
                                                   const float* __restrict__ queries, JoinCopy jc, const float* __restrict__ scale,
                                                   const float* __restrict__ mu_len, SideBound sb, int NQ, int D, bool vec, int rec_cap, const int* __restrict__ start,
                                                   int* __restrict__ q_rec, int* __restrict__ q_rank, int* __restrict__ cnt, int cnt_shift)
{
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    const int sub = threadIdx.x & 7;
    const int q = (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 3);
    const bool valid = q < NQ;
    const size_t at_q = (size_t)(valid ? q : 0);
    const int pieces = (D + 7) >> 3, Dp = pitch - 4;
    uint4 x[NH];
#pragma unroll
    for (int k = 0; k < NH; ++k)
        x[k] = NH * sub + k < pieces ? *reinterpret_cast<const uint4*>(jc.rows + at_q * (size_t)join_pitch(D) + 8 * (NH * sub + k)) : make_uint4(0, 0, 0, 0);
    const float Z = sb.query(jc.norms[at_q], jc.errs[at_q], *scale, *mu_len);
    auto group_sum = [](float t) {                       // the last three steps of the butterfly, over the eight lanes
        t += dpp_f<kDppXor1>(t);
        t += dpp_f<kDppXor2>(t);
        t += dpp_f<kDppHalfMirror>(t);
        return t;
    };
    int cur = start && valid ? start[q] : 0;             // (where the first levels have been taken already: ann_top.hip)
    bool done = !valid;
    for (int step = 0; step <= rec_cap; ++step) {            // a path is never longer than the number of records
        const float* lrow = low + (size_t)(done ? 0 : cur) * (size_t)low_pitch;
        const int4 head = *reinterpret_cast<const int4*>(lrow);
        uint4 n[NH];
#pragma unroll
        for (int k = 0; k < NH; ++k)
            n[k] = NH * sub + k < pieces ? *reinterpret_cast<const uint4*>(lrow + 4 + 4 * (NH * sub + k)) : make_uint4(0, 0, 0, 0);
        float t0 = 0.0f, t1 = 0.0f;
        auto dot = [](uint32_t a, uint32_t b, float c) {
            return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, a), __builtin_bit_cast(f16x2, b), c, false);
        };
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            t0 = dot(n[k].x, x[k].x, t0);
            t1 = dot(n[k].y, x[k].y, t1);
            t0 = dot(n[k].z, x[k].z, t0);
            t1 = dot(n[k].w, x[k].w, t1);
        }
        const float mb = __int_as_float(head.x), t = group_sum(t0 + t1) + mb;
        const bool bucket = head.z < 0;
        bool below = t < 0.0f;
        const bool certain = fabsf(t) > __builtin_fmaf(fabsf(mb), sb.of_offset(), Z);        // (not with a NaN)
        const bool ask = !done && !bucket && !certain;       // (the eight lanes of a query agree)
        if (ballot64(ask) != 0) {
            const float* pl = planes + (size_t)(ask ? cur : 0) * (size_t)pitch;
            const float* xq = queries + at_q * (size_t)D;
            float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
            for (int k = 0; k < kXR; ++k) {
                const int d = 32 * k + 4 * sub;
                const float4 n4 = ask && d < Dp ? *reinterpret_cast<const float4*>(pl + 4 + d) : make_float4(0.f, 0.f, 0.f, 0.f);
                const float4 x4 = ask ? load_piece(xq, d, D, vec) : make_float4(0.f, 0.f, 0.f, 0.f);
                s0 = __builtin_fmaf(n4.x, x4.x, s0);
                s1 = __builtin_fmaf(n4.y, x4.y, s1);
                s2 = __builtin_fmaf(n4.z, x4.z, s2);
                s3 = __builtin_fmaf(n4.w, x4.w, s3);
            }
            const float exact = group_sum((s0 + s1) + (s2 + s3));
            if (ask) below = exact < pl[0];
        }
        if (!done) {
            if (bucket) {
                if (sub == 0) {
                    q_rec[q] = cur;
                    q_rank[q] = atomicAdd(&cnt[cur << cnt_shift], 1);
                }
                done = true;
            } else {
                cur = below ? head.w : head.z;
            }
        }
        if (ballot64(!done) == 0) break;
    }
}

// Scan over the records of the tree in tiles of 1024 (a workgroup each): qoff = exclusive scan of the query counts,
// boff = exclusive scan of the numbers of work items (qb queries each) the buckets need; both get a closing entry at
// index n_rec.  The two sums travel as the halves of one 64-bit value.
typedef unsigned long long u64;
constexpr int kScanTile = 1024;

__device__ __forceinline__ u64 pack_count(int c, int log_qb)
{
    return (u64)(unsigned)c | ((u64)(unsigned)((c + (1 << log_qb) - 1) >> log_qb) << 32);
}
static_assert(kAnnDirect == 16 && kAnnScreen == 32, "log_queries");
__device__ __forceinline__ int log_queries(const AnnForm& form) { return form.screened() ? 5 : 4; }

// exclusive scan of 256 values, one per thread; *total = their sum
__device__ __forceinline__ u64 block_scan_256(u64 v, u64* total, u64* lds4)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    u64 incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) lds4[wave] = incl;
    __syncthreads();
    u64 woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) { const u64 x = lds4[w]; if (w < wave) woff += x; tot += x; }
    __syncthreads();
    *total = tot;
    return woff + incl - v;
}

__global__ __launch_bounds__(256) void k_ann_tile_sums(const int* __restrict__ cnt, int cnt_shift, const int* __restrict__ n_rec_p, int rec_cap,
                                                       u64* __restrict__ tile_sum, AnnForm form)
{
    __shared__ u64 lds4[4];
    const int log_qb = log_queries(form);
    const int n = min(*n_rec_p, rec_cap);
    const int i0 = blockIdx.x * kScanTile + threadIdx.x * 4;
    u64 mine = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) mine += i0 + j < n ? pack_count(cnt[(i0 + j) << cnt_shift], log_qb) : 0ull;
    u64 tot;
    (void)block_scan_256(mine, &tot, lds4);
    if (threadIdx.x == 0) tile_sum[blockIdx.x] = tot;
}

// Second step; also sets the counts back to zero for the next tree.
__global__ __launch_bounds__(256) void k_ann_scan(int* __restrict__ cnt, int cnt_shift, const int* __restrict__ n_rec_p, int rec_cap,
                                                  const u64* __restrict__ tile_sum, int* __restrict__ qoff,
                                                  int* __restrict__ boff, int* __restrict__ n_blocks, AnnForm form)
{
    __shared__ u64 lds4[4];
    const int log_qb = log_queries(form);
    const int n = min(*n_rec_p, rec_cap);
    if (blockIdx.x * kScanTile > n) return;                  // index n itself still gets the closing entries
    u64 before = 0;
    for (int t = threadIdx.x; t < (int)blockIdx.x; t += 256) before += tile_sum[t];
    u64 base;
    (void)block_scan_256(before, &base, lds4);
    const int i0 = blockIdx.x * kScanTile + threadIdx.x * 4;
    u64 v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = i0 + j < n ? pack_count(cnt[(i0 + j) << cnt_shift], log_qb) : 0ull;
    u64 tot;
    u64 run = base + block_scan_256(v[0] + v[1] + v[2] + v[3], &tot, lds4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = i0 + j;
        if (i <= n) {
            qoff[i] = (int)(unsigned)(run & 0xffffffffull);
            boff[i] = (int)(unsigned)(run >> 32);
            if (i == n) *n_blocks = (int)(unsigned)(run >> 32);
            else cnt[i << cnt_shift] = 0;
        }
        run += v[j];
    }
}

// Thread i < NQ puts query i into the list of its bucket; thread i < n_rec writes the descriptors of the work items of
// bucket i: {start and size of the bucket in the tree's permutation, first query in qlist, number of queries}.
__global__ __launch_bounds__(256) void k_ann_fill(int NQ, const int* __restrict__ q_rec, const int* __restrict__ q_rank,
                                                  const int* __restrict__ n_rec_p, int rec_cap, const TreeRec* __restrict__ recs,
                                                  const int* __restrict__ qoff, const int* __restrict__ boff,
                                                  int* __restrict__ qlist, int4* __restrict__ blk_desc, AnnForm form)
{
    const int qb = 1 << log_queries(form);
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < NQ) qlist[qoff[q_rec[i]] + q_rank[i]] = i;
    if (i < min(*n_rec_p, rec_cap)) {
        const int b0 = boff[i], b1 = boff[i + 1];
        if (b1 > b0) {
            const TreeRec rec = recs[i];
            const int q0 = qoff[i], q1 = qoff[i + 1];
            for (int b = b0; b < b1; ++b) {
                const int first = q0 + (b - b0) * qb;
                blk_desc[b] = make_int4(rec.a, rec.b, first, min(qb, q1 - first));
            }
        }
    }
}

__device__ __forceinline__ void chain4(float& acc, const float4& a, const float4& x)
{
    float df;
    df = a.x - x.x; acc = __builtin_fmaf(df, df, acc);
    df = a.y - x.y; acc = __builtin_fmaf(df, df, acc);
    df = a.z - x.z; acc = __builtin_fmaf(df, df, acc);
    df = a.w - x.w; acc = __builtin_fmaf(df, df, acc);
}

// A workgroup takes the work items b = blockIdx.x, + gridDim.x, ...: the bucket and the (up to 16) queries of blk_desc[b].  Per staging step 32 dimensions of up to
// 128 bucket rows and of the 16 query rows pass through LDS; a lane reads "its" bucket rows (two: lane, lane + 64)
// with 16-byte reads and the queries' coordinates as broadcasts.  VEC: D is a multiple of 4 and both matrices are
// 16-byte aligned.
template <int SL, bool VEC>
__global__ __launch_bounds__(256) void k_ann_leaf(const float* __restrict__ points, const float* __restrict__ queries, int D,
                                                  int K, const int* __restrict__ perm, const int4* __restrict__ blk_desc,
                                                  const int* __restrict__ n_blocks, const int* __restrict__ qlist,
                                                  int* __restrict__ q_idx, float* __restrict__ q_dist, AnnForm form)
{
    if (form.screened()) return;
    __shared__ __align__(16) float tile[kCG * kTP];
    __shared__ __align__(16) float xs[kQB * kCH];
    __shared__ int cand[kCG];
    __shared__ int qid_s[kQB];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int n_items = *n_blocks;
    for (int b = blockIdx.x; b < n_items; b += gridDim.x) {
        const int4 desc = blk_desc[b];
        const int start = desc.x, S = desc.y, q0 = desc.z, nq = desc.w;
        if (tid < kQB) qid_s[tid] = qlist[q0 + (tid < nq ? tid : 0)];      // slots beyond nq repeat the first query (ignored later)
        __syncthreads();

        int qid[kQW];
        bool qv[kQW];
        KnnRow<SL> row[kQW];
#pragma unroll
        for (int i = 0; i < kQW; ++i) {
            const int slot = i * 4 + wave;                        // queries are dealt out to the four wavefronts in turn
            qv[i] = slot < nq;
            qid[i] = __builtin_amdgcn_readfirstlane(qid_s[slot]);
            row[i].load(q_idx + (size_t)qid[i] * K, q_dist + (size_t)qid[i] * K, K);
        }
        int n_pass = 0;                                           // pairs of this wavefront that are not above a row's last slot
        const int nqw = (nq - wave + 3) >> 2;                     // queries of this wavefront (0..4), the first nqw slots

        const int piece = tid % kPieces, prow = tid / kPieces;    // staging: kPieces lanes per row
        const bool stage_x = tid < kQB * kPieces;
        const float* xp = queries + (size_t)qid_s[stage_x ? prow : 0] * (size_t)D;
        for (int c0 = 0; c0 < S; c0 += kCG) {
            const int nc = min(kCG, S - c0);
            __syncthreads();                                      // the previous pass is done with cand
            if (tid < kCG) cand[tid] = tid < nc ? perm[start + c0 + tid] : -1;
            __syncthreads();
            const float* rp[kLoads];
            float4 pre[kLoads];
            float4 prex = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                const int rr = prow + kRowsPer * i;
                rp[i] = points + (size_t)cand[rr < nc ? rr : 0] * (size_t)D;       // rows beyond nc repeat row 0 (ignored later)
                pre[i] = load_piece(rp[i], piece * 4, D, VEC);
            }
            if (stage_x) prex = load_piece(xp, piece * 4, D, VEC);
            float acc0[kQW], acc1[kQW];
#pragma unroll
            for (int i = 0; i < kQW; ++i) { acc0[i] = 0.0f; acc1[i] = 0.0f; }
            const bool two = nc > 64;
            for (int d0 = 0; d0 < D; d0 += kCH) {
                __syncthreads();                                  // tile reads of the previous step are done
#pragma unroll
                for (int i = 0; i < kLoads; ++i)
                    *reinterpret_cast<float4*>(&tile[(prow + kRowsPer * i) * kTP + piece * 4]) = pre[i];
                if (stage_x) *reinterpret_cast<float4*>(&xs[prow * kCH + piece * 4]) = prex;
                if (d0 + kCH < D) {
#pragma unroll
                    for (int i = 0; i < kLoads; ++i) pre[i] = load_piece(rp[i], d0 + kCH + piece * 4, D, VEC);
                    if (stage_x) prex = load_piece(xp, d0 + kCH + piece * 4, D, VEC);
                }
                __syncthreads();
                const int pieces = min(kPieces, (D - d0 + 3) >> 2);
                const float* m0 = &tile[lane * kTP];
                const float* m1 = &tile[(lane + 64) * kTP];
                const float* x0 = &xs[wave * kCH];                // slot i * 4 + wave: stride 4 rows
                if (nqw > 2) {
                    for (int p = 0; p < pieces; ++p) {
                        float4 xv[kQW];
#pragma unroll
                        for (int i = 0; i < kQW; ++i) xv[i] = *reinterpret_cast<const float4*>(x0 + i * 4 * kCH + 4 * p);
                        const float4 a0 = *reinterpret_cast<const float4*>(m0 + 4 * p);
#pragma unroll
                        for (int i = 0; i < kQW; ++i) chain4(acc0[i], a0, xv[i]);
                        if (two) {
                            const float4 a1 = *reinterpret_cast<const float4*>(m1 + 4 * p);
#pragma unroll
                            for (int i = 0; i < kQW; ++i) chain4(acc1[i], a1, xv[i]);
                        }
                    }
                } else if (nqw > 0) {
                    for (int p = 0; p < pieces; ++p) {
                        float4 xv[2];
#pragma unroll
                        for (int i = 0; i < 2; ++i) xv[i] = *reinterpret_cast<const float4*>(x0 + i * 4 * kCH + 4 * p);
                        const float4 a0 = *reinterpret_cast<const float4*>(m0 + 4 * p);
#pragma unroll
                        for (int i = 0; i < 2; ++i) chain4(acc0[i], a0, xv[i]);
                        if (two) {
                            const float4 a1 = *reinterpret_cast<const float4*>(m1 + 4 * p);
#pragma unroll
                            for (int i = 0; i < 2; ++i) chain4(acc1[i], a1, xv[i]);
                        }
                    }
                }
            }
            const int c_lo = cand[lane], c_hi = cand[lane + 64];
#pragma unroll
            for (int i = 0; i < kQW; ++i) {
                if (qv[i]) {
                    const bool okv[2] = {lane < nc, two && lane + 64 < nc};
                    const int cv[2] = {c_lo, c_hi};
                    const float dv[2] = {acc0[i], acc1[i]};
                    n_pass += __popcll(ballot64(okv[0] && dv[0] <= row[i].tau)) + __popcll(ballot64(okv[1] && dv[1] <= row[i].tau));
                    row[i].template merge<2>(okv, cv, dv);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < kQW; ++i)
            if (qv[i] && row[i].changed) row[i].store(q_idx + (size_t)qid[i] * K, q_dist + (size_t)qid[i] * K);
        if (form.counts(b) && lane == 0)
            atomicAdd(form.word(b), (unsigned long long)(unsigned)n_pass | (wave == 0 ? (unsigned long long)((unsigned)nq * (unsigned)S) << 32 : 0ull));
        __syncthreads();                                          // done with the ids before the next item's are written
    }
}

// Workgroup q works on query q and the buckets it reached in T trees, wavefront w on those of the trees w, w + 4, ...
// The members of the buckets are gathered in a list, 64 of them at a time get their exact distance (a lane reads "its"
// row, the arithmetic of k_ann_leaf) and are merged into the wavefront's copy of the row; at the end the copies are
// merged.  A row is the K smallest pairs of what it is offered in whatever order, and a pair that a wavefront turns
// away has K pairs below it in that wavefront's row, all of which the final row is offered.
// A query meets a near point in many trees: an id that a wavefront has listed goes into a small direct-mapped table the
// four share, and an id found there is not listed again (whoever put it there evaluates it; an entry that another id has
// overwritten only costs a repeat, which the row turns away).
// Bound by the latency of the gathers: 1,000 queries, 50 trees on 20,000 x 64 clustered points take 48 us here, 23 in each of
// k_planes and k_route (six launches a tree before: 1,780 us).
constexpr int kAnnSeen = 1024;
constexpr int kAnnList = 128;         // of a wavefront: fewer than 64 waiting and up to 64 new ones
// QUADS: how the rows are read (exact_direct; the rule is at the launch).
template <int SL, bool QUADS>
__global__ __launch_bounds__(256) void k_ann_forest(const float* __restrict__ points, const float* __restrict__ queries, int N, int D,
                                                    int K, int T, const int* __restrict__ perm, const int2* __restrict__ reached,
                                                    bool vec_ok, int dpad, int* __restrict__ q_idx, float* __restrict__ q_dist)
{
    // dynamic LDS: the query (dpad) | table (kAnnSeen) | lists (4 x kAnnList) | rows of wavefronts 1..3 (ids, distances)
    extern __shared__ __align__(16) int ann_lds[];
    float* xrow = reinterpret_cast<float*>(ann_lds);
    int* seen = ann_lds + dpad;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int* list = seen + kAnnSeen + wave * kAnnList;
    int* row_i = seen + kAnnSeen + 4 * kAnnList;
    float* row_d = reinterpret_cast<float*>(row_i + 3 * 64 * SL);
    const size_t q = blockIdx.x;
    // (T is at most 64: lane l holds the bucket of tree wave + 4 l)
    const int2 mine = lane < 16 && wave + 4 * lane < T ? reached[q * (size_t)T + (size_t)(wave + 4 * lane)] : make_int2(0, 0);
    for (int d = tid; d < dpad; d += 256) xrow[d] = d < D ? queries[q * (size_t)D + (size_t)d] : 0.0f;
    for (int e = tid; e < kAnnSeen; e += 256) seen[e] = -1;
    KnnRow<SL> row;
    row.load(q_idx + q * (size_t)K, q_dist + q * (size_t)K, K);
    __syncthreads();
    ExploreLds L = {};
    L.xrow = xrow;
    const int n_mine = (T - wave + 3) >> 2;
    // the ids of the next tree travel while those of the present one are worked on
    auto request = [&](int i) {
        const int start = read_lane_i(mine.x, i & 15), size = i < n_mine ? read_lane_i(mine.y, i & 15) : 0;
        return lane < size ? perm[(size_t)(wave + 4 * i) * (size_t)N + (size_t)(start + lane)] : -1;
    };
    int n = 0;
    int next = request(0);
    for (int i = 0; i < n_mine; ++i) {
        const int start = read_lane_i(mine.x, i), size = read_lane_i(mine.y, i);
        const int* ids = perm + (size_t)(wave + 4 * i) * (size_t)N + (size_t)start;
        int id = next;
        next = request(i + 1);
        for (int c0 = 0; c0 < size; c0 += 64) {
            if (c0 > 0) id = c0 + lane < size ? ids[c0 + lane] : -1;
            int* slot = seen + ((uint32_t)id * 2654435761u >> 22);
            const bool list_it = id >= 0 && __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != id;
            const uint64_t m = ballot64(list_it);
            if (list_it) {
                __hip_atomic_store(slot, id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                list[n + mask_prefix(m)] = id;
            }
            n += __popcll(m);
            wave_lds_sync();
            if (n >= 64) {
                exact_direct<SL, QUADS>(L, list, 64, points, D, vec_ok, row);
                n -= 64;
                const int rest = lane < n ? list[64 + lane] : -1;
                wave_lds_sync();
                if (lane < n) list[lane] = rest;
                wave_lds_sync();
            }
        }
    }
    if (n > 0) exact_direct<SL, QUADS>(L, list, n, points, D, vec_ok, row);
    if (wave > 0) {
#pragma unroll
        for (int s = 0; s < SL; ++s) {
            row_i[(wave - 1) * 64 * SL + 64 * s + lane] = row.changed ? row.idx[s] : -1;
            row_d[(wave - 1) * 64 * SL + 64 * s + lane] = row.dist[s];
        }
    }
    __syncthreads();
    if (wave > 0) return;
#pragma unroll 1
    for (int w = 0; w < 3; ++w) {
        bool ok[SL];
        int c[SL];
        float d[SL];
#pragma unroll
        for (int s = 0; s < SL; ++s) {
            c[s] = row_i[w * 64 * SL + 64 * s + lane];
            d[s] = row_d[w * 64 * SL + 64 * s + lane];
            ok[s] = c[s] >= 0;
        }
        row.template merge<SL>(ok, c, d);
    }
    if (row.changed) row.store(q_idx + q * (size_t)K, q_dist + q * (size_t)K);
}

}  // namespace

namespace {

// floats per row of the table of hyperplanes: offset (4 floats) + normal padded to a multiple of 4
int plane_pitch(int D) { return 4 + ((D + 3) & ~3); }
// ... of the rounded ones; 0: not made (see k_route_low).  RSFK_ANN_ROUTE_LOW=1 / 0 says yes or no.  Making them costs with the points,
// what they give comes with the queries and the dimensions (20 trees, without -> with): 300,000 / 300,000 x 128 13.9 -> 13.3 ms, x 50 9.41 -> 9.27,
// x 20 7.66 -> 7.65, x 8 7.67 -> 7.61; 60,000 points, 1M queries x 50 19.1 -> 18.8, x 20 14.8 -> 14.9; 1M points, 100,000 queries x 128
// 20.3 -> 20.0, x 50 13.5 -> 13.6; 50,000 queries and fewer the same.
int low_plane_pitch(int N, int NQ, int D)
{
    if (D > 32 * kXR) return 0;
    const char* e = std::getenv("RSFK_ANN_ROUTE_LOW");
    const bool wanted = e && *e ? e[0] == '1' : NQ >= 100000 && (D > 64 || (D > 32 && (long long)NQ * 4 >= N));
    return wanted ? (16 + 2 * ((D + 7) & ~7) + 63) / 64 * 16 : 0;         // (whole pieces of 64 bytes)
}

// Atomics on one cache line are carried out one after the other, about 14 ns each, and every query is counted by one: with few
// records their counters have lines of their own, as far as 64 K words go (16 K to 1 M: the same).  778,760 queries / 1,370 x 4, 15 trees
// 46.7 -> 13.3 ms, 85,173 / 1,645 x 124, 20 trees 6.0 -> 2.8, 276,641 / 25,337 x 15, 37 trees 12.2 -> 8.4, 500,000 / 100,000 x 40 the same.
// (Which records share a line follows from how a tree is built; that alone has made 8 % of the routing.)
int count_shift(int rec_cap)
{
    int shift = 0;
    while (shift < 5 && ((long long)rec_cap << (shift + 1)) <= 65536) ++shift;
    return shift;
}

}  // namespace

// floats of working memory a record of a tree takes (both tables of hyperplanes)
int ann_plane_pitch(int N, int NQ, int D) { return plane_pitch(D) + low_plane_pitch(N, NQ, D); }
bool ann_low_wanted(int n_trees, int N, int NQ, int D)
{
    const char* e = std::getenv("RSFK_ANN_ROUTE_LOW");
    return low_plane_pitch(N, NQ, D) > 0 && ((e && *e) || ann_copy_pays(n_trees, NQ));
}

size_t ann_ws_ints(int NQ, int rec_cap)
{
    // q_rec | q_rank | qlist (NQ each) | cnt (rec_cap << cnt_shift) | qoff | boff (rec_cap + 1 each) | descriptors of the workgroups
    // (4 ints each, 16-byte aligned) | n_blocks (4) | tile sums
    return (size_t)3 * NQ + ((size_t)rec_cap << count_shift(rec_cap)) + 2 * ((size_t)rec_cap + 1) + 4 + 4 * ((size_t)NQ / kQB + rec_cap + 1) + 4 +
           2 * ((size_t)rec_cap / kScanTile + 2);
}

// The form of a tree's bucket step: the screened one from this share of the pairs downwards, in 1/65536 (kScreenAlways: whatever
// the share, 0: never).  A wavefront has 32 queries to itself there, so that it takes 250,000 queries to fill the device
// (30,000 queries / 20,000 x 100, 20 trees 1.7 -> 2.1 ms) and about 32 of them in a bucket (400,000 / 1M x 50: 19 in a
// bucket of 48, 10 trees 7.2 -> 7.7); in buckets of up to 24 members, where a wavefront of k_ann_leaf has more lanes
// than members, 12 will do (1M / 1M x 16, 20 trees 18.5 -> 13.9, 300,000 / 300,000 x 200 19.7 -> 16.9).  Longer rows make the
// gathers of step 3 dearer: 300,000 / 300,000 x 256 in buckets of 33..66 22.0 -> 22.7 ms, 1M / 1M x 100 78.4 -> 69.6, with the
// line at 20 to 40 % of the pairs alike, 500,000 / 500,000 x 64 13.5 -> 12.1 (20 to 60 % alike), 1M / 60,000 x 8 12.7 -> 9.4
// at 60 % and 9.9 at 20 %.
unsigned int ann_screen_share_q16(int N, int NQ, int D, int K, int n_leaves)
{
    if (K > 64 || D > kAnnScreenDims) return 0;
    double pct = D <= 64 ? 60.0 : 30.0;
    const char* e = std::getenv("RSFK_ANN_SCREEN");             // (read at every call: tests change it)
    if (e && *e) {
        if (e[0] == 'a') return kScreenAlways;
        pct = e[0] >= '0' && e[0] <= '9' ? std::atof(e) : 0.0;
    } else {
        const long long leaves = std::max(n_leaves, 1);
        const bool narrow = (long long)N <= 24 * leaves;
        if (D > 128 + (narrow ? 72 : 0) || NQ < 250000 || (long long)NQ < leaves * (narrow ? 12 : 32)) return 0;
    }
    return (unsigned int)(std::min(100.0, std::max(0.0, pct)) * 65536.0 / 100.0);
}

size_t ann_stat_words(int n_trees) { return (size_t)kAnnStatWords * (size_t)n_trees; }

// First use of a workspace: the bucket counters start at zero (every tree leaves them so), and so do the numbers of pairs.
int launch_ann_ws_init(int* ws, int NQ, int rec_cap, unsigned long long* stats, int n_trees, hipStream_t stream)
{
    const int n_stat = (int)(2 * ann_stat_words(n_trees));
    hipLaunchKernelGGL(k_zero_ints, dim3((unsigned)((n_stat + 255) / 256)), dim3(256), 0, stream, reinterpret_cast<int*>(stats), n_stat);
    int* cnt = ws + (size_t)3 * NQ;
    const int n_cnt = rec_cap << count_shift(rec_cap);
    hipLaunchKernelGGL(k_zero_ints, dim3((unsigned)((n_cnt + 255) / 256)), dim3(256), 0, stream, cnt, n_cnt);
    RSFK_HIP(hipGetLastError());
    return 0;
}

// One tree of the query-set search: routes the queries through the index recs (*n_rec_dev records, at most rec_cap;
// the tree has n_leaves buckets), groups them by bucket and offers the base points perm[..] of the bucket a query
// reached to the query's row.  prev, stats: numbers of pairs of the tree before this one (null: the first) and of this one,
// kAnnStatWords each.  q_copy, p_copy: null, or the copy of the queries, of the points
// (with q_copy only: the screened bucket step reads them).  n_trees: of the call.  start: the records from which the queries go on (null: the root).  ws: ann_ws_ints(NQ, rec_cap) ints, prepared by launch_ann_ws_init; planes: rec_cap
// ann_plane_pitch(N, NQ, D) floats and 256 bytes.
int launch_ann_tree(const float* points, const float* queries, int N, int NQ, int D, int K, const int* perm, const TreeRec* recs,
                    const int* n_rec_dev, int rec_cap, int n_leaves, const JoinCopy* q_copy, const JoinCopy* p_copy,
                    int n_trees, const int* start, int* ws, float* planes, int* q_idx, float* q_dist,
                    const unsigned long long* prev, unsigned long long* stats, hipStream_t stream)
{
    if (NQ <= 0) return 0;
    RSFK_CHECK(K >= 1 && K <= kMaxK, "query-set search: K must be in 1..1024");
    RSFK_CHECK(recs != nullptr && rec_cap >= 1, "query-set search: the tree has no index");
    int* q_rec = ws;
    int* q_rank = q_rec + NQ;
    int* qlist = q_rank + NQ;
    int* cnt = qlist + NQ;
    const int cnt_shift = count_shift(rec_cap);
    int* qoff = cnt + ((size_t)rec_cap << cnt_shift);
    int* boff = qoff + rec_cap + 1;
    int4* blk_desc = reinterpret_cast<int4*>(ws + (((boff + rec_cap + 1) - ws + 3) & ~(ptrdiff_t)3));
    int* n_blocks = reinterpret_cast<int*>(blk_desc + ((size_t)NQ / kQB + rec_cap + 1));
    u64* tile_sum = reinterpret_cast<u64*>(ws + ((ann_ws_ints(NQ, rec_cap) - 2 * ((size_t)rec_cap / kScanTile + 2)) & ~(size_t)1));
    const int pitch = plane_pitch(D), low_pitch = q_copy ? low_plane_pitch(N, NQ, D) : 0;
    float* low = low_pitch ? reinterpret_cast<float*>((reinterpret_cast<uintptr_t>(planes + (size_t)rec_cap * (size_t)pitch) + 255) & ~(uintptr_t)255) : nullptr;
    hipLaunchKernelGGL(k_planes, dim3((unsigned)((rec_cap + 3) / 4)), dim3(256), 0, stream, points, D, recs, n_rec_dev, rec_cap, planes,
                       pitch, low, low_pitch, low ? q_copy->mu : nullptr, low ? q_copy->scale() : nullptr);
    const unsigned g_route = (unsigned)(((size_t)NQ * 8 + 255) / 256);
    const bool vec_q = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(queries) & 15) == 0;
    if (low && D <= 64)
        hipLaunchKernelGGL(k_route_low<1>, dim3(g_route), dim3(256), 0, stream, planes, pitch, low, low_pitch, queries, *q_copy, q_copy->scale(),
                           q_copy->mu_len(), SideBound(D), NQ, D, vec_q, rec_cap, start, q_rec, q_rank, cnt, cnt_shift);
    else if (low)
        hipLaunchKernelGGL(k_route_low<2>, dim3(g_route), dim3(256), 0, stream, planes, pitch, low, low_pitch, queries, *q_copy, q_copy->scale(),
                           q_copy->mu_len(), SideBound(D), NQ, D, vec_q, rec_cap, start, q_rec, q_rank, cnt, cnt_shift);
    else if (vec_q)
        hipLaunchKernelGGL((k_route<true, false>), dim3(g_route), dim3(256), 0, stream, planes, pitch, queries, NQ, D, recs, rec_cap,
                           start, q_rec, q_rank, cnt, cnt_shift, nullptr);
    else
        hipLaunchKernelGGL((k_route<false, false>), dim3(g_route), dim3(256), 0, stream, planes, pitch, queries, NQ, D, recs, rec_cap,
                           start, q_rec, q_rank, cnt, cnt_shift, nullptr);
    // a bucket with c queries takes ceil(c / 16) work items: at most NQ / 16 + (buckets with queries) in all
    const int most_items = NQ / kQB + std::min(n_leaves, NQ) + 1;
    const unsigned int share_q16 = ann_screen_share_q16(N, NQ, D, K, n_leaves);
    AnnForm form = {share_q16 != 0 ? prev : nullptr, stats, share_q16, p_copy ? ann_half_share_q16(N, NQ, D, n_trees, share_q16) : 0u, 0};
    while ((most_items >> form.shift) > 512) ++form.shift;
    const unsigned g_scan = (unsigned)(rec_cap / kScanTile + 1);
    hipLaunchKernelGGL(k_ann_tile_sums, dim3(g_scan), dim3(256), 0, stream, cnt, cnt_shift, n_rec_dev, rec_cap, tile_sum, form);
    hipLaunchKernelGGL(k_ann_scan, dim3(g_scan), dim3(256), 0, stream, cnt, cnt_shift, n_rec_dev, rec_cap, tile_sum, qoff, boff, n_blocks, form);
    const unsigned g_fill = (unsigned)((std::max(NQ, rec_cap) + 255) / 256);
    hipLaunchKernelGGL(k_ann_fill, dim3(g_fill), dim3(256), 0, stream, NQ, q_rec, q_rank, n_rec_dev, rec_cap, recs, qoff, boff, qlist,
                       blk_desc, form);
    // (the forms that are not taken find out in every workgroup, hence few of them)
    if (form.prev && form.half_q16 != 0 &&
        launch_ann_screen_half(*q_copy, *p_copy, points, queries, D, K, perm, blk_desc, n_blocks, most_items, qlist, q_idx, q_dist, form, stream))
        return 1;
    if (form.prev && form.half_q16 != form.share_q16) {
        if (launch_ann_screen(points, queries, D, K, perm, blk_desc, n_blocks, most_items, qlist, q_idx, q_dist, form, stream)) return 1;
    }
    const unsigned g_leaf = (unsigned)std::min(most_items, kLeafGrid);
    const bool vec = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) | reinterpret_cast<uintptr_t>(queries)) & 15) == 0;
#define RSFK_ANN_CASE(SLV)                                                                                                   \
    {                                                                                                                        \
        if (vec)                                                                                                             \
            hipLaunchKernelGGL((k_ann_leaf<SLV, true>), dim3(g_leaf), dim3(256), 0, stream, points, queries, D, K, perm,       \
                               blk_desc, n_blocks, qlist, q_idx, q_dist, form);                                        \
        else                                                                                                                 \
            hipLaunchKernelGGL((k_ann_leaf<SLV, false>), dim3(g_leaf), dim3(256), 0, stream, points, queries, D, K, perm,       \
                               blk_desc, n_blocks, qlist, q_idx, q_dist, form);                                        \
    }
    if (K <= 64) RSFK_ANN_CASE(1)
    else if (K <= 128) RSFK_ANN_CASE(2)
    else if (K <= 256) RSFK_ANN_CASE(4)
    else if (K <= 512) RSFK_ANN_CASE(8)
    else RSFK_ANN_CASE(16)
#undef RSFK_ANN_CASE
    RSFK_HIP(hipGetLastError());
    return 0;
}

size_t ann_forest_lds(int D, int K) { return sizeof(int) * ((size_t)((D + 31) & ~31) + kAnnSeen + 4 * kAnnList + (size_t)6 * 64 * row_slots(K)); }

// Trees of a batch of nb that are searched together (0: one tree after the other).  Together, a query gathers the rows of its
// buckets by itself, up to NQ MAX D floats a tree; one after the other, up to 16 queries of a bucket share them, at the price
// of six launches a tree.  Time of the search, one after the other -> together (uniform points where nothing is said):
//   20,000 x 64 clustered, buckets of up to 34, 50 trees: 1,000 queries 1.78 -> 0.09 ms, 10,000 1.99 -> 0.44, 40,000 3.59 -> 1.59
//   1M x 100, up to 66, 50 trees: 2,000 queries (1.3e7 floats) 3.5 -> 1.8 ms, 20,000 (1.3e8) 8.7 -> 9.0, 100,000 16 -> 40
//   100,000 x 100, up to 66, 50 trees: 10,000 queries (6.6e7) 2.90 -> 2.93 ms, 50,000 5.1 -> 14.2
//   300,000 x 8, up to 18, 50 trees: 200,000 queries (2.9e7) 10.2 -> 4.7 ms;  5,000 x 129, K = 300, 9 trees: 600 queries (4.7e7)
//   4.0 -> 1.1;  70,000 x 784, K = 90, 10 trees: 10,000 queries (1.4e9) 2.8 -> 10.1
// Repeated points make buckets far above MAX.  Up to kAnnSeen members the table of the ids a query has met spares it the same
// rows in every tree (20,000 x 64 in groups of 200 equal rows, 50 trees, 1,000 queries 2.08 -> 0.10 ms).  Beyond that it gathers
// them T times, and about NQ max_bucket / N queries do so, against one workgroup that takes the whole bucket for 16 of
// them: 20,000 points, half of them equal, 6 trees, x 16: 8,000 queries 2.3 -> 1.4 ms, 16,000 2.9 -> 2.5;  x 64: 2,000 queries
// 3.6 -> 2.9, 4,000 3.8 -> 5.9;  x 200: 1,000 queries 9.5 -> 6.3, 2,000 9.0 -> 15.4;  60,000 x 64, a tenth equal: 8,000 queries
// 2.55 -> 2.56, 16,000 2.5 -> 4.0.  The two are alike at NQ max_bucket / N x D of 0.9e5 to 1.8e5.
int ann_forest_group(int N, int NQ, int D, int K, int MAX, int max_bucket, int rec_cap, int nb)
{
    const char* e = std::getenv("RSFK_ANN_FOREST");
    if (e && e[0] == '0') return 0;
    if (nb < 2 || ann_forest_lds(D, K) > (size_t)64 << 10) return 0;
    const bool forced = e && e[0] == '1';
    constexpr double kMostFloats = 5e7, kMostHot = 1.2e5;
    if (!forced && (double)NQ * (double)MAX * (double)D > kMostFloats) return 0;
    if (!forced && max_bucket > kAnnSeen && (double)NQ * (double)max_bucket * (double)D > kMostHot * (double)N) return 0;
    // hyperplanes and buckets reached: 1 GB at most
    const size_t per_tree = sizeof(float) * (size_t)rec_cap * (size_t)ann_plane_pitch(N, NQ, D) + sizeof(int2) * (size_t)NQ;
    const int group = (int)std::min<size_t>((size_t)std::min(nb, 64), ((size_t)1 << 30) / per_tree);
    return group >= 2 ? group : 0;
}

// The search in T trees at once.  recs, n_rec_dev, perm: those of the first tree, the others follow (n_rec_dev: kTreeStatPitch apart); planes: T rec_cap
// ann_plane_pitch(N, NQ, D) floats; reached: 2 NQ T ints.
int launch_ann_forest(const float* points, const float* queries, int N, int NQ, int D, int K, int T, const int* perm, const TreeRec* recs,
                      const int* n_rec_dev, int rec_cap, float* planes, int* reached, int* q_idx, float* q_dist, hipStream_t stream)
{
    RSFK_CHECK(K >= 1 && K <= kMaxK && T >= 1 && T <= 64, "query-set search: out of range");
    RSFK_CHECK(recs != nullptr && rec_cap >= 1, "query-set search: the tree has no index");
    int2* where = reinterpret_cast<int2*>(reached);
    const int pitch = plane_pitch(D);
    hipLaunchKernelGGL(k_planes, dim3((unsigned)((rec_cap + 3) / 4), (unsigned)T), dim3(256), 0, stream, points, D, recs, n_rec_dev, rec_cap,
                       planes, pitch, nullptr, 0, nullptr, nullptr);
    const dim3 g_route((unsigned)(((size_t)NQ * 8 + 255) / 256), (unsigned)T);
    const bool vec_q = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(queries) & 15) == 0;
    if (vec_q)
        hipLaunchKernelGGL((k_route<true, true>), g_route, dim3(256), 0, stream, planes, pitch, queries, NQ, D, recs, rec_cap, nullptr,
                           nullptr, nullptr, nullptr, 0, where);
    else
        hipLaunchKernelGGL((k_route<false, true>), g_route, dim3(256), 0, stream, planes, pitch, queries, NQ, D, recs, rec_cap, nullptr,
                           nullptr, nullptr, nullptr, 0, where);
    const bool vec_p = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(points) & 15) == 0;
    const int dpad = (D + 31) & ~31;
    const size_t lds = ann_forest_lds(D, K);
    // Rows of a few lines in an L2 are read sooner by a lane each: four lanes that exchange what they load take more instructions, and save
    // requests that only count where there are many, from farther away.  A call, own rows -> quads, K = 16, 50 trees, 10,000 queries: 5,000 x 24 +7 %, x 48 -1,
    // x 60 -7, x 96 -14; 20,000 x 40 -2; 40,000 x 24 +2, x 32 -4, x 48 -9, x 96 -16; 300,000 x 24 -1, x 32 -2; K = 32, 20 trees, 23,234 queries: 367,009 x 29 (clusters) -17; 1,000 x 64 0; K = 10, 12 trees, 10,000 queries: 5,000 x 24 +4, x 72 +3, 3,000 x 150 -6; K = 16, 20
    // trees, 8,000 queries: 3,000 x 56 +4, 20,000 x 56 -4, 20,000 x 112 -14; K = 10, 20 trees: 2,000 x 100 +3 to +5; K = 107, 50 trees, 62,271 queries: 1,909 x 3 +29.
    const size_t words = (size_t)N * (size_t)D;
    const bool quads = D > 128 || (D > 48 && T * K >= 250 && words >= (size_t)1 << 18) || (D >= 28 && T * K >= 500 && words >= (size_t)1 << 20);
#define RSFK_ANN_CASE(SLV)                                                                                                    \
    do {                                                                                                                     \
        auto* kernel = quads ? k_ann_forest<SLV, true> : k_ann_forest<SLV, false>;                                            \
        hipLaunchKernelGGL(kernel, dim3((unsigned)NQ), dim3(256), lds, stream, points, queries, N, D, K, T, perm, where, vec_p, dpad, \
                           q_idx, q_dist);                                                                                   \
    } while (0)
    switch (row_slots(K)) {
    case 1: RSFK_ANN_CASE(1); break;
    case 2: RSFK_ANN_CASE(2); break;
    case 4: RSFK_ANN_CASE(4); break;
    case 8: RSFK_ANN_CASE(8); break;
    default: RSFK_ANN_CASE(16); break;
    }
#undef RSFK_ANN_CASE
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
