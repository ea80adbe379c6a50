// Random-sample tree building for a batch of trees, level-synchronous.
//
// Replaces the reference's per-level kernel chain of
// RSFK::create_bucket_from_sample_tree (src/rsfk.cu:500-1207):
// build_tree_init, build_tree_check_active_points, build_tree_check_points_side,
// build_tree_count_new_nodes, build_tree_accumulate_child_count,
// build_tree_organize_sample_candidates, build_tree_create_nodes,
// build_tree_update_parents, build_tree_post_update_parents, build_tree_utils,
// build_tree_fix, build_tree_max_leaf_size, build_tree_set_leaves_idx and
// build_tree_bucket_points (src/kernels/build_tree_*.cu, create_node.cu).
//
// Representation: every tree keeps a permutation of 0..N-1 in which each node
// is a contiguous segment; splitting a node is a stable partition of its
// segment (left members first).  There are no per-point parent/depth arrays
// and no per-point atomics.
//
//   wide phase : nodes larger than `small` points.  Each level is three
//                launches over all trees of the batch: (1) hyperplane + side
//                test + per-chunk left counts, (2) stable scatter with
//                wave64 ballot / mbcnt ranks, child creation by the chunk-0
//                workgroup of each node, (3) chunk bookkeeping for the next
//                level.
//   middle phase: with few points (small inputs, few trees) nodes of up to some
//                thousand points are split down to `small` by one workgroup
//                each (k_mid), which replaces most of the wide levels.
//
//   tail phase : one workgroup finishes the whole subtree of a node with at
//                most `small` points inside LDS (all the re-draw levels that
//                the min/max rule causes touch only such nodes).
//
//   chain phase : nodes of some hundred points are finished from the distances of
//                their points (k_chain).
//
// Arithmetic follows the reference bit for bit: the hyperplane offset and the
// side test are sums of 32 lane-strided partials combined by the xor butterfly
// (create_node.cu:122-135, build_tree_check_points_side.cu:131-149); a half
// wavefront plays the role of the 32-lane warp.
#include "rsfk_common.hpp"
#include "wave64.hpp"
#include "knn_list.hpp"
#include "bf16.hpp"
#include "tree_sweep.hpp"
#include "mfma_split.hpp"
#include "level_notes.hpp"
#include <vector>
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <chrono>

namespace rsfk {

namespace {

constexpr int kBlock = 256;


// Counters of a batch.  Those of the queue of level l are in entry l & 3, so that a level can be queued on the stream before
// the one before it has run.
struct LevelCounters {
    struct alignas(8) Queue {
        int nodes;     // nodes of a wide level
        int chunks;    // and their chunks
    } queue[4];
    int n_tail;        // tail tasks appended so far
    int n_mid;         // ... and tasks of the middle phase
    int n_mid_next[2]; // ... of its second and its third launch
    int n_chain;       // nodes for the chain phase appended so far, at the front of their queue
    int n_chain_back;  // ... and at its back: those that are hardly split in vain
    int overflow;      // set when a queue capacity is exceeded
    // time spent in the three steps of the wide levels (hyperplanes, side tests, scatter) and in the tail, in ticks of
    // the device's constant-rate clock: the first thread of a kernel that opens a step closes the one before it
    long long last_tick;
    long long phase_ticks[4];
    // nodes of the chain phase taken from the queue, beyond the first one of every workgroup: node i belongs to share i % kShares
    // (additions to one cache line come one after the other)
    static constexpr int kShares = 16;
    struct alignas(128) Share { int taken; } share[kShares];
};

// Counts for the report of a build (how many points the side tests of all levels looked at, and how many of them
// the screen left to the exact test): kStatSlots slots a cache line apart, so that the workgroups' additions do not
// all go to one address; slot s holds [points, undecided points] at stat[kStatPitch * s + 0 / 1].
constexpr int kStatSlots = 64, kStatPitch = 32;
__device__ __forceinline__ void stat_add(unsigned long long* stat, int slot, int which, int v)
{
    if (stat && v) atomicAdd(&stat[kStatPitch * (slot & (kStatSlots - 1)) + which], (unsigned long long)v);
}

// ended: the step that ends where the calling kernel begins (-1: none, the clock is only started)
__device__ __forceinline__ void phase_tick(LevelCounters* ctr, int ended)
{
    const long long now = (long long)wall_clock64();
    if (ended >= 0 && ctr->last_tick != 0) ctr->phase_ticks[ended] += now - ctr->last_tick;
    ctr->last_tick = now;
}

// ---------------------------------------------------------------------------
// helpers
// ---------------------------------------------------------------------------

// Length of a normal in LDS: zero padded to whole 16-byte pieces of either screening copy.
__host__ __device__ inline int nvec_len(int D) { return (D + 15) & ~15; }

// Hyperplane of (x1,x2) by one wavefront (all 64 lanes call): normal into LDS nvec[0..nvec_len(D)), and
// hp[0] = offset (order of create_node.cu:122-135: 32 lane-strided partial sums + xor butterfly),
// hp[1] = the length L of the normal that the 8-bit rows' bounds are for (kNormalLeast added: bf16.hpp), hp[2] = the sum of its components (any
// order: only the screens use them, with a margin).  The sum of squares in it is used where the squares neither underflow nor overflow.  A pair with the same coordinates has the normal 0 and every point on its left (0 < 0):
// its hp[1] is kZeroNormal, which makes the bounds of the screens negative, so that no point is left to the exact test
// (100,000 x 32, a tenth of the points in groups of 2,000 equal rows, 10 trees: 947 -> 220 ms).
// SCREEN8 false: hp[1] is the 1-norm, of which the bfloat16 screen takes the sign (tail of 3,000 x 9000 22.0 ms with the sum of squares, 21.8 without, of 1,200 x 20000 89.7 and 88.4).
constexpr float kZeroNormal = -1e30f;
template <bool SCREEN8 = true>
__device__ __forceinline__ void make_hyperplane_wave(const float* __restrict__ x1, const float* __restrict__ x2,
                                                     int D, float* nvec, float* hp)
{
    const int lane = lane_id();
    const int Dn = nvec_len(D);
    const int hl = lane & 31;
    const bool lowh = lane < 32;
    // Both halves of the wavefront walk the dimensions hl, hl + 32, ... (the loads of eight steps are requested
    // together): the lower half forms the offset with the arithmetic of create_node.cu:122-135, the normal
    // and the sum of its squares, the upper half the 1-norm and the sum of the components.
    float s = 0.0f, s2 = 0.0f;
    for (int d0 = hl; d0 < D; d0 += 256) {
        float t1[8], t2[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int d = d0 + 32 * k;
            t1[k] = d < D ? x1[d] : 0.0f;
            t2[k] = d < D ? x2[d] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int d = d0 + 32 * k;
            if (d < D) {
                const float nd = t1[k] - t2[k];
                if (lowh) {
                    nvec[d] = nd;
                    const float prod = nd * (t1[k] + t2[k]);
                    s = s + prod * 0.5f;
                    if (SCREEN8) s2 = __builtin_fmaf(nd, nd, s2);
                } else {
                    s += fabsf(nd);
                    s2 += nd;
                }
            }
        }
    }
    for (int d = D + lane; d < Dn; d += 64) nvec[d] = 0.0f;
    s = half_butterfly_sum(s);
    s2 = half_butterfly_sum(s2);
    const float sq = SCREEN8 ? read_lane_f(s2, 0) : 0.0f;
    if (lane == 0) hp[0] = s;
    if (lane == 32) {
        const float l2 = __builtin_sqrtf(sq * (kRmsShare * kRmsShare * 1.0005f * (float)D));
        hp[1] = s == 0.0f ? kZeroNormal : (SCREEN8 && s > 1e-9f ? fminf(s, l2) : s) + kNormalLeast;
        hp[2] = s2;
    }
}

// Screen of the side test for eight points per wavefront (right = n.x < b): lanes 8g..8g+7 work on
// the point of group g; all lanes of a group return its answer.  (With the 8-bit copy and short rows a group may
// be LPP = 4 or 2 lanes: 16 or 32 points per wavefront.)
//
// The decision is always the one of the exact fp32 test (resolve_exact below: 32 lane-strided fused
// multiply-add chains + xor butterfly, build_tree_check_points_side.cu:131-149), but most points never
// touch their fp32 row: a bfloat16 copy of the row (half the bytes) gives an approximate n.x together
// with S~ = sum |n_d||x~_d|.  bfloat16 keeps 8 significant bits: rounding x to x~ (round to nearest)
// changes n.x by at most 2^-8 sum |n_d||x_d| <= 2^-8 (1+2^-7) S~, and the fp32 summations of the two
// paths are off by at most (D/8 + D/32 + 16) 2^-24 S~ together, so whenever |approx - b| exceeds
// `band` * S~ (band = 1.01 (2^-8 (1+2^-7) + (D/8 + D/32 + 16) 2^-24), computed by the caller) the sign of
// (n.x - b) is the same for the exact evaluation: right[u] is final.  Otherwise (a few per cent of the
// points; also NaN or infinite values, and every point when there is no bfloat16 copy) redo[u] is set and
// the caller hands the point to resolve_exact.
//
// NB points per group are handled per call, so that NB row gathers per lane are in flight before the
// first is needed (the loop over points is bound by the latency of these gathers otherwise).
//
// With the 8-bit copy (bf16.hpp) the row is 16 header bytes + one byte per coordinate: approx = lo sum_d n_d +
// scale sum_d n_d q_d, undecided band e1 L(n) (hp1 = L(n), hp2 = sum of the components of the
// normal of the point's node).  Only lane 0 of a group holds the header, so only its right / redo are meaningful
// (with either copy the callers use lane 0 only).
// (KU: pieces of a row a lane has in flight, 8-bit copy)
// INSIDE: the header comes with the row, as its first piece, above nothing of the normal (header_inside says where; 16 floats that can be read have to be before
// nvec0): the row then comes in loads of whole lines, each once, where a load of its own asks for the first line again while it is on its way.  Middle phase
// of 123,457 x 37, 12 trees 0.202 -> 0.182 ms, of 3,000 x 200, 10 trees 0.046 -> 0.043.  In the tail kernel, which is bound by its instructions, only where the row is
// then a single step of its lanes (up to 16 dimensions: 458,955 x 15, 27 trees 1.77 -> 1.65 ms, 1M x 2, 10 trees 1.48 -> 1.43); with longer rows it is the same, and to decide it at each row
// costs 1 to 3 % (5,000 x 24, 50 trees 135 -> 138 us, 8,000 x 32, 8 trees 114 -> 117, 5,000 x 52, 50 trees 156 -> 160, 200,000 x 32, 12 trees 363 -> 367).
template <int LPP>
bool header_inside(int D) { return (q8_padded(D) >> 4) % LPP != 0; }      // (the last step has a lane to spare)

template <int NB, bool Q8, int LPP = 8, int KU = 1, bool INSIDE = false>
__device__ __forceinline__ void side_screen8(const float* nvec0, int nstride, const int (&j)[NB], const float (&b)[NB],
                                             const float (&hp1)[NB], const float (&hp2)[NB],
                                             const uint16_t* __restrict__ pb16, const uint8_t* __restrict__ q8,
                                             const int (&id)[NB], int D, float band,
                                             const bool (&valid)[NB], bool (&right)[NB], bool (&redo)[NB])
{
    if (Q8) {
        static_assert(LPP == 8 || LPP == 4 || LPP == 2, "lanes per point");
        const int sub = lane_id() & (LPP - 1);
#pragma unroll
        for (int u = 0; u < NB; ++u) { right[u] = false; redo[u] = valid[u]; }
        const size_t pitch = (size_t)q8_pitch(D);
        const int pieces = (q8_padded(D) >> 4) + (INSIDE ? 1 : 0);
        if (!INSIDE) q8 += 16;
        else nvec0 -= 16;
        float da[NB];
        uint4 head[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            da[u] = 0.0f;
            head[u] = make_uint4(0u, 0u, 0u, 0u);
            if (!INSIDE && valid[u] && sub == 0) head[u] = *reinterpret_cast<const uint4*>(q8 - 16 + (size_t)id[u] * pitch);
        }
        for (int k0 = sub; k0 < pieces; k0 += KU * LPP) {
            uint4 w[KU][NB];
#pragma unroll
            for (int y = 0; y < KU; ++y)
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    w[y][u] = make_uint4(0u, 0u, 0u, 0u);
                    if (valid[u] && (KU == 1 || k0 + y * LPP < pieces))
                        w[y][u] = *reinterpret_cast<const uint4*>(q8 + (size_t)id[u] * pitch + 16 * (k0 + y * LPP));
                }
#pragma unroll
            for (int y = 0; y < KU; ++y) {
                const int k = k0 + y * LPP;
                if (KU > 1 && k >= pieces) break;
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    const float* nvec = nvec0 + (size_t)j[u] * nstride + 16 * k;
                    const uint32_t ww[4] = {w[y][u].x, w[y][u].y, w[y][u].z, w[y][u].w};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float4 nq = *reinterpret_cast<const float4*>(&nvec[4 * q]);
                        da[u] = __builtin_fmaf(nq.x, (float)((ww[q] >> 0) & 0xffu), da[u]);
                        da[u] = __builtin_fmaf(nq.y, (float)((ww[q] >> 8) & 0xffu), da[u]);
                        da[u] = __builtin_fmaf(nq.z, (float)((ww[q] >> 16) & 0xffu), da[u]);
                        da[u] = __builtin_fmaf(nq.w, (float)((ww[q] >> 24) & 0xffu), da[u]);
                    }
                    if (INSIDE && y == 0 && k == 0) { head[u] = w[0][u]; da[u] = 0.0f; }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            float d = da[u];
            d += dpp_f<kDppXor1>(d);
            if (LPP >= 4) d += dpp_f<kDppXor2>(d);
            if (LPP >= 8) d += dpp_f<kDppHalfMirror>(d);
            const float lo = __uint_as_float(head[u].y), scale = __uint_as_float(head[u].z), e1 = __uint_as_float(head[u].w);
            const float approx = __builtin_fmaf(scale, d, lo * hp2[u]);
            const bool certain = fabsf(approx - b[u]) > e1 * hp1[u];       // false if anything is NaN
            right[u] = approx < b[u];
            redo[u] = valid[u] && !certain;
        }
        return;
    }
    // hyperplane of point u of this group: normal nvec0 + j[u] * nstride, offset b[u] (groups may differ)
    const int lane = lane_id();
    const int sub = lane & 7;
#pragma unroll
    for (int u = 0; u < NB; ++u) { right[u] = false; redo[u] = valid[u]; }
    (void)hp2;
    if (pb16 != nullptr) {
        const int Dv = bf16_valid(D);
        const size_t pitch = (size_t)bf16_pitch(D);
        float da[NB], sa[NB];
#pragma unroll
        for (int u = 0; u < NB; ++u) { da[u] = 0.0f; sa[u] = 0.0f; }
        for (int e = sub * 8; e < Dv; e += 64) {
            uint4 w[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                w[u] = make_uint4(0u, 0u, 0u, 0u);
                if (valid[u]) w[u] = *reinterpret_cast<const uint4*>(pb16 + (size_t)id[u] * pitch + e);
            }
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const float* nvec = nvec0 + (size_t)j[u] * nstride;
                const float4 n0 = *reinterpret_cast<const float4*>(&nvec[e]);
                const float4 n1 = *reinterpret_cast<const float4*>(&nvec[e + 4]);
                const uint32_t ww[4] = {w[u].x, w[u].y, w[u].z, w[u].w};
                const float nn[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float x0 = __uint_as_float(ww[q] << 16);
                    const float x1 = __uint_as_float(ww[q] & 0xffff0000u);
                    da[u] = __builtin_fmaf(nn[2 * q], x0, da[u]);
                    da[u] = __builtin_fmaf(nn[2 * q + 1], x1, da[u]);
                    sa[u] = __builtin_fmaf(fabsf(nn[2 * q]), fabsf(x0), sa[u]);
                    sa[u] = __builtin_fmaf(fabsf(nn[2 * q + 1]), fabsf(x1), sa[u]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            // sum over the 8 lanes of the group (any order will do for the screen)
            float d = da[u], a = sa[u];
            d += dpp_f<kDppXor1>(d); d += dpp_f<kDppXor2>(d); d += dpp_f<kDppHalfMirror>(d);
            a += dpp_f<kDppXor1>(a); a += dpp_f<kDppXor2>(a); a += dpp_f<kDppHalfMirror>(a);
            // (a below 1e38: no partial sum of the exact test overflows)
            const bool certain = fabsf(d - b[u]) > a * band + (1e-30f + fminf(hp1[u], 0.0f)) && a < 1e38f;
            right[u] = d < b[u];
            redo[u] = valid[u] && !certain;
        }
    }
}

// Exact side tests for the points the screen could not decide: n.x by one half wavefront (32 lanes, lane hl
// runs the chain over d = hl, hl + 32, ...; the loads of a chain are issued eight at a time), then the xor butterfly.  list[i] = position of the
// point (local to the caller) | slot of its node << 16.  One half wavefront per point, two points per half
// wavefront at a time so that their row loads overlap; all threads of the workgroup call.  id_at(pos) gives the
// point, apply(pos, right) receives the answer in lane 0 of the half wavefront.
// (h of `halves`: which half wavefront of those that work on the list this is)
template <typename Entry, typename IdAt, typename Apply>
__device__ __forceinline__ void resolve_exact(int halves, int h, const Entry* list, int n, const float* nvec0, int nstride, const float* b_of,
                                              const float* __restrict__ points, int D, IdAt id_at, Apply apply)
{
    const int hl = threadIdx.x & 31;
    for (int base = 0; base < n; base += 2 * halves) {
        const int ia = base + h, ib = base + halves + h;
        const bool va = ia < n, vb = ib < n;
        const int ea = va ? list[ia] : 0, eb = vb ? list[ib] : 0;
        const float* xa = points + (size_t)id_at(ea & 0xffff) * D;
        const float* xb = points + (size_t)id_at(eb & 0xffff) * D;
        const float* na = nvec0 + (size_t)(ea >> 16) * nstride;
        const float* nb = nvec0 + (size_t)(eb >> 16) * nstride;
        float sa = 0.0f, sb = 0.0f;
        for (int d0 = hl; d0 < D; d0 += 256) {
            float xv[8], yv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                xv[k] = (va && d0 + 32 * k < D) ? xa[d0 + 32 * k] : 0.0f;
                yv[k] = (vb && d0 + 32 * k < D) ? xb[d0 + 32 * k] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (d0 + 32 * k < D) {
                    sa = __builtin_fmaf(na[d0 + 32 * k], xv[k], sa);
                    sb = __builtin_fmaf(nb[d0 + 32 * k], yv[k], sb);
                }
            }
        }
        sa = half_butterfly_sum(sa);
        sb = half_butterfly_sum(sb);
        if (hl == 0) {
            if (va) apply(ea & 0xffff, sa < b_of[ea >> 16]);
            if (vb) apply(eb & 0xffff, sb < b_of[eb >> 16]);
        }
    }
}

constexpr int kWideChunk = 1024;     // points per workgroup in the wide passes (the side tests keep a chunk's undecided points in LDS)
constexpr int kSideBatch = 4;        // points per group and call of the screen in the wide phase

// The queues nodes go to: the next wide level (entry `slot` of the counters) and the tail kernel (one workgroup per node).
struct NodeQueues {
    TreeNode* next;
    int next_cap, chunk_cap, slot;
    TreeNode* tail;      // (or the middle phase)
    int tail_cap;
    LevelCounters* ctr;
    int* n_tail;         // its counter
};

// Append the nc children of a node to their queues; a node of the next wide level is given its chunks too.  at[i]: place
// of child i in the queue of the next wide level, or -1.  (All workgroups of a level add to the same few words, one
// after the other: a queue is one addition for both children, and for its nodes and chunks together.)
__device__ __forceinline__ void emit_children(const TreeNode (&c)[2], int nc, const TreeParams& P, const NodeQueues& Q, int (&at)[2])
{
    bool wide[2], forced[2];
    int chunks[2], n_wide = 0, n_chunks = 0, n_tail = 0;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        forced[i] = c[i].depth >= P.MAX_DEPTH - 1;
        wide[i] = i < nc && !c[i].leaf && !forced[i] && c[i].count > P.small;
        chunks[i] = wide[i] ? (c[i].count + P.chunk - 1) / P.chunk : 0;
        n_wide += wide[i] ? 1 : 0;
        n_chunks += chunks[i];
        n_tail += i < nc && !wide[i] ? 1 : 0;
        at[i] = -1;
    }
    int next = 0, chunk = 0, tail = 0;
    if (n_wide) {
        const unsigned long long was = atomicAdd(reinterpret_cast<unsigned long long*>(&Q.ctr->queue[Q.slot]),
                                                 (unsigned long long)(unsigned)n_wide | ((unsigned long long)(unsigned)n_chunks << 32));
        next = (int)(unsigned)was;
        chunk = (int)(unsigned)(was >> 32);
    }
    if (n_tail) tail = atomicAdd(Q.n_tail, n_tail);
    if ((n_wide && (next + n_wide > Q.next_cap || chunk + n_chunks > Q.chunk_cap)) || (n_tail && tail + n_tail > Q.tail_cap)) {
        Q.ctr->overflow = 1;
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (i >= nc) continue;
        TreeNode t = c[i];
        if (wide[i]) {
            t.chunk0 = chunk;
            chunk += chunks[i];
            at[i] = next;
            Q.next[next++] = t;
        } else {
            if (forced[i]) t.leaf = 1;
            Q.tail[tail++] = t;
        }
    }
}

// The split / min-size-merge / leaf rules for a node whose left side has `a`
// members (src/kernels/build_tree_update_parents.cu:64-75,106-134).  Returns the
// number of children written to c0, c1.
__device__ __forceinline__ int split_rules(const TreeNode& nd, int a, int MIN, int MAX, int child_buf,
                                           TreeNode& c0, TreeNode& c1)
{
    const int r = nd.count - a;
    const uint64_t kl = child_key(nd.key, 0), kr = child_key(nd.key, 1);
    c0.tree = c1.tree = nd.tree;
    c0.depth = c1.depth = nd.depth + 1;
    c0.buf = c1.buf = child_buf;
    c0.rec = c1.rec = 0;
    c0.chunk0 = c1.chunk0 = 0;
    if (a == 0 || r == 0) {
        c0.start = nd.start; c0.count = nd.count; c0.dstart = nd.start; c0.dcount = nd.count;
        c0.key = a ? kl : kr; c0.leaf = nd.count <= MAX - 2;
        return 1;
    }
    if (min(a, r) < MIN) {
        const bool left_big = a >= r;
        c0.start = nd.start; c0.count = nd.count;
        c0.dstart = left_big ? nd.start : nd.start + a;
        c0.dcount = left_big ? a : r;
        c0.key = left_big ? kl : kr; c0.leaf = nd.count <= MAX;
        return 1;
    }
    c0.start = nd.start; c0.count = a; c0.dstart = nd.start; c0.dcount = a;
    c0.key = kl; c0.leaf = a <= MAX - 2;
    c1.start = nd.start + a; c1.count = r; c1.dstart = nd.start + a; c1.dcount = r;
    c1.key = kr; c1.leaf = r <= MAX - 2;
    return 2;
}

// Index of the tree (TreeRec): reserve the records of the children of node nd and write nd's own record.
// recs / n_rec belong to the tree of nd.  p1, p2: the drawn pair.  A node with one child (an empty side, or the
// min-size merge) routes every query the same way: it leaves no record and its child takes over its place, so a
// tree has fewer than twice as many records as buckets whatever its depth.
__device__ __forceinline__ void index_split(TreeRec* recs, int* n_rec, int rec_cap, int my_rec, int p1, int p2, int nc,
                                            int& rec0, int& rec1, LevelCounters* ctr)
{
    if (nc != 2) {
        rec0 = rec1 = my_rec;
        return;
    }
    const int base = atomicAdd(n_rec, 2);
    rec0 = base;
    rec1 = base + 1;
    if (base + 2 <= rec_cap && my_rec < rec_cap) {
        TreeRec r;
        r.a = p1; r.b = p2; r.c0 = rec0; r.c1 = rec1;
        recs[my_rec] = r;
    } else {
        ctr->overflow = 1;
    }
}

__device__ __forceinline__ void index_bucket(TreeRec* recs, int rec_cap, int my_rec, int start, int count, LevelCounters* ctr)
{
    if (my_rec < rec_cap) {
        TreeRec r;
        r.a = start; r.b = count; r.c0 = -1; r.c1 = -1;
        recs[my_rec] = r;
    } else {
        ctr->overflow = 1;
    }
}

// ---------------------------------------------------------------------------
// wide phase kernels
// ---------------------------------------------------------------------------

// One per tree of the batch, each in cache lines of its own: the workgroups of all trees add to them at the same time, and additions
// to one line are carried out one after the other (chain phase of 50 trees of 20,000 x 64 points, with an index: 321 us with all trees
// in a few lines, 207 so).  The extremes, which every node of the chain phase reads, wait for those additions where they share their line
// (chain phase of one tree of 1M x 64, buckets of 8..16, 1.39 -> 0.37 ms, of 16 trees of 62,500 x 64 0.28 -> 0.20).
struct alignas(4 * kTreeStatPitch) TreeStats {
    int n_leaves;           // buckets of at most kBucketSplit points, stored from the front of the leaf table
    int n_big;              // larger buckets, stored from the back of the leaf table
    int n_rec;              // records of the index, when one is written
    alignas(128) int levels;        // (read far more often than written: not in the line that is added to)
    int max_leaf;
    int min_leaf;
};

// A batch begins: permutations, counters, and the root of every tree (workgroup 0).
__global__ __launch_bounds__(256) void k_tree_init(int* __restrict__ perm, NodeQueues Q, TreeParams P, int B, int seed0, int* pmap,
                                                   TreeStats* __restrict__ stats, unsigned long long* __restrict__ stat)
{
    const size_t total = (size_t)P.N * (size_t)B;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x)
        perm[i] = (int)(i % (size_t)P.N);
    if (blockIdx.x != 0) return;
    for (int i = threadIdx.x; i < (int)(sizeof(LevelCounters) / sizeof(int)); i += 256) reinterpret_cast<int*>(Q.ctr)[i] = 0;
    for (int i = threadIdx.x; i < kStatSlots * kStatPitch; i += 256) stat[i] = 0ull;
    __threadfence();
    __syncthreads();
    const int t = threadIdx.x;
    if (t >= B) return;
    TreeStats s;
    s.n_leaves = 0; s.n_big = 0; s.levels = 0; s.max_leaf = 0; s.min_leaf = 0x7fffffff;
    s.n_rec = 1;                           // record 0 is the root
    stats[t] = s;
    TreeNode r;
    r.tree = t; r.start = 0; r.count = P.N; r.dstart = 0; r.dcount = P.N; r.depth = 0; r.buf = 0; r.leaf = 0;
    r.rec = 0; r.chunk0 = 0;
    r.key = root_key(seed0 + t);
    // the root is never a leaf (src/kernels/build_tree_init.cu:79) unless the depth limit forces it
    const TreeNode c[2] = {r, r};
    int at[2];
    emit_children(c, 1, P, Q, at);
    if (pmap) pmap[t * pm::kPaths] = at[0];      // path 0 of level 0 = the root, if it is split at all
}

// bytes of a node's record for k_side_q8: [scale of the second part, 128 x it x (254 sum m1 + sum m2), bound of the residuals, 0 | first part | second part]
__host__ __device__ inline size_t side_op_bytes(int D) { return 16 + 2 * (size_t)q8_pitch(D); }

// A wide level begins: hyperplanes of its nodes, one wavefront per node -- record ni of the table is
// [offset, L(n) (bf16.hpp), sum of the components, 0 | normal, nvec_len(D) floats]; the workgroups of a node (one per
// chunk, up to a thousand at the first levels) fetch the record instead of each making the hyperplane again --, the
// chunks of the nodes, and the level's counts for the host, which has queued this level from bounds on them.
__global__ __launch_bounds__(256) void k_level_planes(const float* __restrict__ points, TreeParams P,
                                                      const int* __restrict__ perm0, const int* __restrict__ perm1,
                                                      const TreeNode* __restrict__ nodes, int level, int node_cap,
                                                      float* __restrict__ table, uint8_t* __restrict__ ops, int* __restrict__ chunk2node,
                                                      LevelCounters* ctr, unsigned long long* __restrict__ stat, LevelNote* note, int seq)
{
    extern __shared__ __align__(16) float lds_p[];          // per wavefront: 4 + nvec_len(D) floats
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n_nodes = min(ctr->queue[level & 3].nodes, node_cap);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        phase_tick(ctr, 2);
        ctr->queue[(level + 1) & 3].nodes = 0;                   // (of the level before the last two: nobody needs it any more)
        const int n_chunks = ctr->queue[level & 3].chunks;
        ctr->queue[(level + 1) & 3].chunks = 0;
        note->n_nodes = n_nodes;
        note->n_chunks = n_chunks;
        note->n_tail = P.mid ? ctr->n_mid : ctr->n_tail;
        note->overflow = ctr->overflow;
        __hip_atomic_store(&note->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const int ni = blockIdx.x * (blockDim.x >> 6) + wave;
    if (ni >= n_nodes) return;
    const int rec = 4 + nvec_len(P.D);
    float* mine = lds_p + (size_t)wave * rec;
    const TreeNode nd = nodes[ni];
    for (int k = lane; k * P.chunk < nd.count; k += 64) chunk2node[nd.chunk0 + k] = ni;
    if (lane == 0) stat_add(stat, ni, 0, nd.count);
    const int* perm = (nd.buf ? perm1 : perm0) + (size_t)nd.tree * (size_t)P.N;
    int r1, r2;
    pick_pair(nd.key, nd.dcount, r1, r2);
    const int p1 = perm[nd.dstart + r1] & kIdMask;
    const int p2 = perm[nd.dstart + r2] & kIdMask;
    if (lane == 0) mine[3] = 0.0f;
    make_hyperplane_wave(points + (size_t)p1 * P.D, points + (size_t)p2 * P.D, P.D, mine + 4, mine);
    wave_lds_sync();
    float* out = table + (size_t)ni * rec;
    for (int i = lane; i < rec; i += 64) out[i] = mine[i];
    if (!ops) return;
    // operand rows of k_side_q8: the two 8-bit parts of the normal, byte for byte below a row of the 8-bit copy (zeros below its header)
    float most = 0.0f;
    for (int d = lane; d < P.D; d += 64) most = fmaxf(most, fabsf(mine[4 + d]));
    const pm::NormalParts parts(wave_max(most));
    const int pitch = q8_pitch(P.D);
    uint8_t* op = ops + (size_t)ni * side_op_bytes(P.D);
    float rs = 0.0f;
    int M = 0;
    for (int at = 4 * lane; at < pitch; at += 256) {
        uint32_t w1 = 0u, w2 = 0u;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int d = at + k - 16;
            if (d >= 0 && d < P.D) {
                int i1, i2;
                rs += parts.split(mine[4 + d], i1, i2);
                M += 254 * i1 + i2;
                w1 |= (uint32_t)(i1 & 0xff) << (8 * k);
                w2 |= (uint32_t)(i2 & 0xff) << (8 * k);
            }
        }
        *reinterpret_cast<uint32_t*>(op + 16 + at) = w1;
        *reinterpret_cast<uint32_t*>(op + 16 + pitch + at) = w2;
    }
    rs = pm::wave_sum_f(rs);
    M = wave_sum_i(M);
    if (lane == 0)
        *reinterpret_cast<float4*>(op) = make_float4(parts.s2, parts.s2 * (128.0f * (float)M), pm::NormalParts::residual(rs, mine[1]), 0.0f);
}

// Side test of one chunk of one node: sets bit 31 of the permutation entry of
// every member on the right side and counts the members on the left.  (By the bfloat16 copy, or by the fp32 rows alone; with the 8-bit copy
// k_side_q8 takes its place.)
__global__ __launch_bounds__(kBlock) void k_side(const float* __restrict__ points, const uint16_t* __restrict__ pb16,
                                                 TreeParams P,
                                                 int* __restrict__ perm0, int* __restrict__ perm1,
                                                 const TreeNode* __restrict__ nodes, int slot, LevelCounters* ctr,
                                                 const int* __restrict__ chunk2node, int* __restrict__ chunk_left,
                                                 const float* __restrict__ planes, unsigned long long* __restrict__ stat)
{
    extern __shared__ __align__(16) float side_lds[];      // record of the node's hyperplane (k_level_planes)
    float* hp_s = side_lds;                                 // offset, L(n) (bf16.hpp), sum of the components
    float* nvec = side_lds + 4;                             // nvec_len(D) floats
    __shared__ int left_s, n_def_s;
    __shared__ int deferred[1024];                          // points of the chunk left to the exact test (chunk <= 1024)
    const int c = blockIdx.x;
    if (c >= ctr->queue[slot].chunks) return;
    if (c == 0 && threadIdx.x == 0) phase_tick(ctr, 0);
    const int ni = chunk2node[c];
    const TreeNode nd = nodes[ni];
    const int k = c - nd.chunk0;
    int* perm = (nd.buf ? perm1 : perm0) + (size_t)nd.tree * (size_t)P.N;
    if (threadIdx.x == 0) { left_s = 0; n_def_s = 0; }
    {
        const int rec4 = (4 + nvec_len(P.D)) >> 2;          // 16-byte pieces of the record
        const float4* src = reinterpret_cast<const float4*>(planes + (size_t)ni * (size_t)(4 * rec4));
        for (int i = threadIdx.x; i < rec4; i += kBlock) reinterpret_cast<float4*>(side_lds)[i] = src[i];
    }
    __syncthreads();
    const float b = hp_s[0], n1 = hp_s[1], sn = hp_s[2];
    const int pos0 = nd.start + k * P.chunk;
    const int pos1 = min(nd.start + nd.count, pos0 + P.chunk);
    constexpr int kGroupsL = kBlock / 8;                             // groups of eight lanes, one point each
    const int grp = threadIdx.x >> 3, sub8 = threadIdx.x & 7;
    const int iters = (pos1 - pos0 + kGroupsL - 1) / kGroupsL;
    int lefts = 0;
    for (int it = 0; it < iters; it += kSideBatch) {
        int id[kSideBatch], jz[kSideBatch], pos[kSideBatch];
        float bb[kSideBatch], h1[kSideBatch], h2[kSideBatch];
        bool valid[kSideBatch], right[kSideBatch], redo[kSideBatch];
#pragma unroll
        for (int u = 0; u < kSideBatch; ++u) {
            pos[u] = pos0 + (it + u) * kGroupsL + grp;
            valid[u] = pos[u] < pos1;
            id[u] = valid[u] ? (perm[pos[u]] & kIdMask) : 0;
            jz[u] = 0;
            bb[u] = b;
            h1[u] = n1;
            h2[u] = sn;
        }
        side_screen8<kSideBatch, false>(nvec, 0, jz, bb, h1, h2, pb16, nullptr, id, P.D, P.band, valid, right, redo);
#pragma unroll
        for (int u = 0; u < kSideBatch; ++u) {
            if (valid[u] && sub8 == 0) {
                if (redo[u]) {
                    deferred[atomicAdd(&n_def_s, 1)] = pos[u] - pos0;
                } else {
                    perm[pos[u]] = right[u] ? (id[u] | (int)0x80000000) : id[u];
                    lefts += right[u] ? 0 : 1;
                }
            }
        }
    }
    __syncthreads();
    resolve_exact(kBlock >> 5, (int)threadIdx.x >> 5, deferred, n_def_s, nvec, 0, hp_s, points, P.D,
                  [&](int local) { return perm[pos0 + local] & kIdMask; },
                  [&](int local, bool right) {
                      const int id = perm[pos0 + local] & kIdMask;
                      perm[pos0 + local] = right ? (id | (int)0x80000000) : id;      // build_tree_check_points_side.cu:149
                      lefts += right ? 0 : 1;
                  });
    if (lefts) atomicAdd(&left_s, lefts);
    __syncthreads();
    if (threadIdx.x == 0) {
        chunk_left[c] = left_s;
        stat_add(stat, c, 1, n_def_s);
    }
}

// The same by the 8-bit copy.  What bounds it is the rows, a cache line or more each from anywhere in the copy: the device delivers 55 to 59 G
// lines a second, 6.3 TB/s of rows of several lines.  So that nothing else does, a wavefront has 64 rows on their way at a time, their places are
// known before the first is asked for, no line of a short row is asked for twice (a load takes lines, and the headers come with them), and the products come from
// the matrix cores: all points of a chunk meet the same hyperplane, whose two 8-bit parts (pm::NormalParts) are rows of one operand; the bytes of the
// points' rows as they lie in memory, header and all, above zeros of the normal, are columns of the other.
//   LINE false, rows of 64 bytes: a load is 16 rows, lane (row % 16, piece / 16) has a piece of 16 bytes.  Even and odd rows of the first operand repeat
//   the two parts, so every lane holds both sums of row lane % 16 of each of four tiles.
//   LINE true, longer rows: a load is 128 bytes of 8 rows, so columns 0..7 of the operand are the even pieces of the eight rows and 8..15 the odd ones; rows 4 i,
//   4 i + 1 of the first operand are the parts below even pieces, 4 i + 2, 4 i + 3 those below odd ones, and a row's sums are added up over lanes c and c + 8.
// Either way lane l then decides point l of the 64.  A level of 1M x 100, 50 trees: 1.49 -> 0.99 ms, of 10M x 32, 10 trees: 2.53 -> 2.15, of 1M x 256, 20 trees:
// 1.52 -> 1.31 (a few per cent of it by the tighter bound of bf16.hpp), against eight (or two) lanes per point that multiply byte by byte, two vector instructions
// each, and ask for a point's place, its row and its header in turn.  Headers by loads of their own: 1.11, 2.38; rows on multiples of 128 bytes: 1.35 for 256 dimensions.
struct SideLds {                                            // besides the record of the hyperplane
    float4 head[kBlock / 64][64];
    int ids[kWideChunk];                                    // members of the chunk, bit 31 as it will be stored
    uint16_t undecided[kWideChunk];
    int left, n_undecided;
};
constexpr size_t kSideRecordMost = (size_t)160 * 1024 - sizeof(SideLds);      // bytes of the record (D up to 38,384)

template <bool LINE>
__global__ __launch_bounds__(kBlock) void k_side_q8(const float* __restrict__ points, const uint8_t* __restrict__ q8, TreeParams P,
                                                    int* __restrict__ perm0, int* __restrict__ perm1,
                                                    const TreeNode* __restrict__ nodes, int slot, LevelCounters* ctr,
                                                    const int* __restrict__ chunk2node, int* __restrict__ chunk_left,
                                                    const float* __restrict__ planes, const uint8_t* __restrict__ ops,
                                                    unsigned long long* __restrict__ stat)
{
    extern __shared__ __align__(16) float side_lds[];      // record of the node's hyperplane (k_level_planes)
    constexpr int kRounds = kWideChunk / kBlock;
    constexpr int kTiles = LINE ? 8 : 4, kRows = 64 / kTiles;       // of the 64 points of a wavefront; lanes of a row
    __shared__ SideLds own;
    int* ids = own.ids;
    uint16_t* undecided = own.undecided;
    const int c = blockIdx.x;
    if (c >= ctr->queue[slot].chunks) return;
    if (c == 0 && threadIdx.x == 0) phase_tick(ctr, 0);
    const int ni = chunk2node[c];
    const TreeNode nd = nodes[ni];
    const int tid = threadIdx.x, lane = tid & 63, row = lane % kRows, piece = lane / kRows;
    int* perm = (nd.buf ? perm1 : perm0) + (size_t)nd.tree * (size_t)P.N;
    const int pos0 = nd.start + (c - nd.chunk0) * kWideChunk;
    const int n = min(nd.start + nd.count - pos0, kWideChunk);
    int id[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r) id[r] = r * kBlock + tid < n ? (perm[pos0 + r * kBlock + tid] & kIdMask) : 0;
    const float* rec = planes + (size_t)ni * (size_t)(4 + nvec_len(P.D));
    for (int i = tid; i < (4 + nvec_len(P.D)) >> 2; i += kBlock)
        reinterpret_cast<float4*>(side_lds)[i] = reinterpret_cast<const float4*>(rec)[i];
    if (tid == 0) { own.left = 0; own.n_undecided = 0; }
    const float b = rec[0], length = rec[1], sum = rec[2];
    const size_t pitch = (size_t)q8_pitch(P.D);
    const uint8_t* op = ops + (size_t)ni * side_op_bytes(P.D);
    const float4 scales = *reinterpret_cast<const float4*>(op);
    const int below_at = 16 * (LINE ? 2 * (lane >> 4) + ((lane >> 1) & 1) : lane >> 4);
    const uint8_t* part = op + 16 + (lane & 1) * pitch + below_at;
    const int steps = LINE ? (int)((pitch + 127) >> 7) : 1;
    float4* heads = own.head[tid >> 6];
    pm::v4i normal = *reinterpret_cast<const pm::v4i*>(part);       // of the first step, which is the only one of most rows
    __syncthreads();
    int lefts = 0;
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
        if (r * kBlock + (tid & ~63) >= n) break;
        const uint8_t* src[kTiles];
        pm::v4i acc[kTiles], w[kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            src[t] = q8 + (size_t)__shfl(id[r], kRows * t + row, 64) * pitch + 16 * piece;
            w[t] = *reinterpret_cast<const pm::v4i*>(src[t]);
            acc[t] = pm::v4i{0, 0, 0, 0};
        }
        if (piece == 0) {
#pragma unroll
            for (int t = 0; t < kTiles; ++t) *reinterpret_cast<pm::v4i*>(&heads[kRows * t + row]) = w[t];
        }
        pm::v4i below = normal;
        for (int k = 1;; ++k) {
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
                acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(below, w[t] ^ (int)0x80808080, acc[t], 0, 0, 0);
            if (!LINE || k >= steps) break;
            below = pm::v4i{0, 0, 0, 0};
            if (128 * k + below_at < (int)pitch) below = *reinterpret_cast<const pm::v4i*>(part + 128 * k);
#pragma unroll
            for (int t = 0; t < kTiles; ++t)
                if (128 * k + 16 * piece < (int)pitch) w[t] = *reinterpret_cast<const pm::v4i*>(src[t] + 128 * k);
        }
        int i1 = 0, i2 = 0;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            int s1 = acc[t][0], s2 = acc[t][1];
            if (LINE) {
                s1 = lane & 8 ? acc[t][2] : s1;
                s2 = lane & 8 ? acc[t][3] : s2;
                s1 += dpp_i<kDppRor8>(s1);
                s2 += dpp_i<kDppRor8>(s2);
            }
            i1 = piece == t ? s1 : i1;
            i2 = piece == t ? s2 : i2;
        }
        wave_lds_sync();
        const float4 head = heads[lane];
        const float lo = head.y, scale = head.z, e1 = head.w;
        const float product = __builtin_fmaf(scales.x, __builtin_fmaf(254.0f, (float)i1, (float)i2), scales.y);
        const float approx = __builtin_fmaf(scale, product, lo * sum);
        const float band = __builtin_fmaf(e1, length, (fabsf(lo) + 255.0f * scale) * scales.z);
        const bool valid = r * kBlock + tid < n;
        const bool certain = fabsf(approx - b) > band;                     // false if anything is NaN
        const bool right = certain && approx < b;
        ids[r * kBlock + tid] = right ? id[r] | (int)0x80000000 : id[r];
        lefts += valid && certain && !right ? 1 : 0;
        if (valid && !certain) undecided[atomicAdd(&own.n_undecided, 1)] = (uint16_t)(r * kBlock + tid);
        wave_lds_sync();
    }
    __syncthreads();
    resolve_exact(kBlock >> 5, tid >> 5, undecided, own.n_undecided, side_lds + 4, 0, side_lds, points, P.D,
                  [&](int local) { return ids[local] & kIdMask; },
                  [&](int local, bool right) {
                      if (right) ids[local] |= (int)0x80000000;            // build_tree_check_points_side.cu:149
                      lefts += right ? 0 : 1;
                  });
    lefts = wave_sum_i(lefts);
    if (lane == 0 && lefts) atomicAdd(&own.left, lefts);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
        if (r * kBlock + tid < n) perm[pos0 + r * kBlock + tid] = ids[r * kBlock + tid];
    if (tid == 0) {
        chunk_left[c] = own.left;
        stat_add(stat, c, 1, own.n_undecided);
    }
}

// Stable scatter of one chunk into the other permutation buffer; the workgroup
// of chunk 0 also applies the split rules and appends the children.
__global__ __launch_bounds__(kBlock) void k_scatter(TreeParams P, int* __restrict__ perm0, int* __restrict__ perm1,
                                                    const TreeNode* __restrict__ nodes, int slot,
                                                    const int* __restrict__ chunk2node, const int* __restrict__ chunk_left,
                                                    NodeQueues Q, TreeRec* __restrict__ recs, TreeStats* stats,
                                                    int rec_cap, int2* __restrict__ child)
{
    LevelCounters* ctr = Q.ctr;
    __shared__ int red[2][kBlock / 64];
    const int c = blockIdx.x;
    if (c >= ctr->queue[slot].chunks) return;
    if (c == 0 && threadIdx.x == 0) phase_tick(ctr, 1);
    const int ni = chunk2node[c];
    const TreeNode nd = nodes[ni];
    const int first = nd.chunk0;
    const int nch = (nd.count + P.chunk - 1) / P.chunk;
    const int k = c - first;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    const size_t toff = (size_t)nd.tree * (size_t)P.N;
    const int* src = (nd.buf ? perm1 : perm0) + toff;
    int* dst = (nd.buf ? perm0 : perm1) + toff;
    const int pos0 = nd.start + k * P.chunk;
    const int pos1 = min(nd.start + nd.count, pos0 + P.chunk);
    // rounds of four entries per thread (entry u of a thread at r0 + u kBlock + tid: loads and stores stay coalesced,
    // four loads in flight, one exchange of the wavefronts' counts per round); the entries of the first round (the
    // only one with chunks of 1024) are requested before the counts of the node's chunks are added up, so that the
    // two trips to memory go side by side
    constexpr int kPer = 4;
    int v[kPer];
    auto request = [&](int r0) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int pos = r0 + u * kBlock + tid;
            v[u] = pos < pos1 ? src[pos] : -1;            // (beyond the chunk: counts as a right one, is not stored)
        }
    };
    request(pos0);

    // lefts in the chunks before this one, and in the whole node
    int before = 0, all = 0;
    for (int j = tid; j < nch; j += kBlock) {
        const int x = chunk_left[first + j];
        all += x;
        if (j < k) before += x;
    }
    before = wave_sum_i(before);
    all = wave_sum_i(all);
    if (lane == 0) { red[0][wave] = before; red[1][wave] = all; }
    __syncthreads();
    before = 0; all = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) { before += red[0][w]; all += red[1][w]; }

    int lbase = before;                                   // lefts of the node before the current round
    __shared__ int wcnt4[kPer][kBlock / 64];
    for (int r0 = pos0; r0 < pos1; r0 += kPer * kBlock) {
        if (r0 > pos0) request(r0);
        uint64_t m[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            m[u] = ballot64(v[u] >= 0);
            if (lane == 0) wcnt4[u][wave] = __popcll(m[u]);
        }
        __syncthreads();
        int run = lbase;                                  // lefts before entry (u, wavefront 0)
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            int woff = 0, tot = 0;
#pragma unroll
            for (int w = 0; w < kBlock / 64; ++w) { const int x = wcnt4[u][w]; if (w < wave) woff += x; tot += x; }
            const int pos = r0 + u * kBlock + tid;
            if (pos < pos1) {
                const int lrank = run + woff + mask_prefix(m[u]);      // lefts of the node before this position
                const bool right = v[u] < 0;
                const int dest = right ? nd.start + all + (pos - nd.start) - lrank : nd.start + lrank;
                dst[dest] = v[u] & kIdMask;
            }
            run += tot;
        }
        lbase = run;
        __syncthreads();
    }
    if (k == 0 && tid == 0) {
        TreeNode c[2];
        const int nc = split_rules(nd, all, P.MIN, P.MAX, nd.buf ^ 1, c[0], c[1]);
        if (recs) {
            int r1, r2;
            pick_pair(nd.key, nd.dcount, r1, r2);
            index_split(recs + (size_t)nd.tree * rec_cap, &stats[nd.tree].n_rec, rec_cap, nd.rec, src[nd.dstart + r1] & kIdMask,
                        src[nd.dstart + r2] & kIdMask, nc, c[0].rec, c[1].rec, ctr);
        }
        int at[2];
        emit_children(c, nc, P, Q, at);
        // where the members of either side are at the next level (a node with one child keeps them together)
        if (child) child[ni] = make_int2(at[0], nc == 2 ? at[1] : at[0]);
    }
}

// What k_side_q8 leaves behind, from sides that are already known (one bit per point of the tree, pm::k_pm_sweep and
// pm::k_pm_resolve): bit 31 of the permutation entries of a chunk and the number of its left members.
__global__ __launch_bounds__(kBlock) void k_pm_mark(TreeParams P, int* __restrict__ perm0, int* __restrict__ perm1,
                                                    const TreeNode* __restrict__ nodes, const int* __restrict__ n_chunks,
                                                    const int* __restrict__ chunk2node, int* __restrict__ chunk_left,
                                                    const uint32_t* __restrict__ sidebits, int W)
{
    __shared__ int part[kBlock / 64];
    const int c = blockIdx.x;
    if (c >= *n_chunks) return;
    const int ni = chunk2node[c];
    const TreeNode nd = nodes[ni];
    const int k = c - nd.chunk0;
    int* perm = (nd.buf ? perm1 : perm0) + (size_t)nd.tree * (size_t)P.N;
    const uint32_t* bits = sidebits + (size_t)nd.tree * (size_t)W;
    const int pos0 = nd.start + k * P.chunk;
    const int pos1 = min(nd.start + nd.count, pos0 + P.chunk);
    int lefts = 0;
    for (int r0 = pos0; r0 < pos1; r0 += 4 * kBlock) {
        int id[4];
        uint32_t w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int pos = r0 + u * kBlock + (int)threadIdx.x;
            id[u] = pos < pos1 ? (perm[pos] & kIdMask) : -1;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) w[u] = id[u] >= 0 ? bits[id[u] >> 5] : 0u;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int pos = r0 + u * kBlock + (int)threadIdx.x;
            if (id[u] >= 0) {
                const bool right = (w[u] >> (id[u] & 31)) & 1u;
                perm[pos] = right ? (id[u] | (int)0x80000000) : id[u];
                lefts += right ? 0 : 1;
            }
        }
    }
    lefts = wave_sum_i(lefts);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = lefts;
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 0;
#pragma unroll
        for (int i = 0; i < kBlock / 64; ++i) all += part[i];
        chunk_left[c] = all;
    }
}

// ---------------------------------------------------------------------------
// tail phase: one workgroup per small node, whole subtree in LDS
// ---------------------------------------------------------------------------
struct SmallNode {
    int start, count, dstart, dcount;     // offsets inside the task's segment
    int depth;
    int rec;                              // record of the node in the index of the tree, if one is written
    int vain;                             // tail phase: splits in vain just before this node
    int place;                            // tail phase, nodes for the chain phase: place among those of its end of the queue
    uint64_t key;
};

// Entry of the leaf table that the `at`-th bucket of its kind takes: small buckets fill the table of the tree from the
// front, large ones from the back, so that each kind can be handed to its own kernel as a plain (start, size) array.
__device__ __forceinline__ void store_leaf(int tree, int gstart, int count, int at, int leaf_cap,
                                           int* __restrict__ leaf_start, int* __restrict__ leaf_size, LevelCounters* ctr)
{
    if (at < leaf_cap) {
        const int slot = count > kBucketSplit ? leaf_cap - 1 - at : at;
        leaf_start[(size_t)tree * leaf_cap + slot] = gstart;
        leaf_size[(size_t)tree * leaf_cap + slot] = count;
    } else {
        ctr->overflow = 1;
    }
}

// One bucket straight to the table (nodes that became buckets in the wide phase).
__device__ __forceinline__ void emit_leaf(int tree, int gstart, int count, int depth, int leaf_cap,
                                          int* __restrict__ leaf_start, int* __restrict__ leaf_size,
                                          TreeStats* stats, LevelCounters* ctr)
{
    TreeStats* st = stats + tree;
    const int at = atomicAdd(count > kBucketSplit ? &st->n_big : &st->n_leaves, 1);
    store_leaf(tree, gstart, count, at, leaf_cap, leaf_start, leaf_size, ctr);
    atomicMax(&st->levels, depth + 1);
    atomicMax(&st->max_leaf, count);
    atomicMin(&st->min_leaf, count);
}

// Is a node of `count` points likely to be split in vain many times in a row?  A split counts when both sides have at least MIN points,
// which leaves count - 2 MIN + 1 of the places it may have.
__device__ __forceinline__ bool often_in_vain(int count, int MIN) { return 8 * (count - 2 * MIN + 1) <= count; }

constexpr int kTailMost = 2048;      // points of the largest node the tail kernel takes
constexpr int kVainMost = 4;         // splits in vain in a row after which a node leaves for the chain phase
constexpr int kMaxGroup = 16;        // nodes of one level of a subtree worked on together

// One workgroup finishes the subtree of a task level by level: the nodes of a level are taken kMaxGroup (or
// fewer, G) at a time -- their hyperplanes are made together (one wavefront each), all their points are tested in
// one sweep, and each node is partitioned by one wavefront -- so the number of dependent trips to memory per
// subtree is a few per level instead of a few per node.
// TB = threads per workgroup: 256, or 512 / 1024 for launches over so few subtrees that workgroups of 256 would leave
// most of the device idle (the phases of a level then have more lanes).  CHAIN: nodes of at most P.chain_max points go
// to the queue of the chain phase; otherwise those of them that have been split in vain kVainMost times in a row.  The form of 256 threads is for many subtrees and lives by six wavefronts per SIMD, for which
// it has to stay within 80 registers (81 and five wavefronts: 1M x 100, 50 trees 10.8 -> 12.3 ms).
// LPP: lanes per point in the screen (side_screen8), eight with the bfloat16 copy; KU: 16-byte pieces of a point's row each of them has in
// flight.
template <bool Q8, int TB, bool CHAIN, int LPP, int KU, bool INSIDE>
__global__ __launch_bounds__(TB, CHAIN ? 4 : 6) void k_tail(const float* __restrict__ points,
                                                 const uint16_t* __restrict__ pb16, const uint8_t* __restrict__ q8, TreeParams P,
                                                 const int* __restrict__ perm0, const int* __restrict__ perm1,
                                                 int* __restrict__ perm_out,
                                                 const TreeNode* __restrict__ tasks, int n_tasks, int leaf_most, int node_most, int G,
                                                 int leaf_cap, int* __restrict__ leaf_start, int* __restrict__ leaf_size,
                                                 TreeStats* stats, LevelCounters* ctr,
                                                 TreeRec* __restrict__ recs_all, int rec_cap,
                                                 unsigned long long* __restrict__ stat, TreeNode* __restrict__ chain_all, int chain_cap)
{
    // dynamic LDS: seg[small] | tmp[small] | nvec[G][nvec_len(D)] | lrec[leaf_most] | level lists 2 x node_most |
    // nodes for the chain phase [node_most] | fmap[small]
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int Dv = nvec_len(P.D);
    int* seg = reinterpret_cast<int*>(lds_raw);
    int* tmp = seg + P.small;
    float* nvec = reinterpret_cast<float*>(tmp + P.small);
    // buckets of this subtree, written to the table of the tree together at the end (one reservation per
    // workgroup instead of one atomic round trip per bucket): x = start, y = size | rank among its kind << 16
    int2* lrec = reinterpret_cast<int2*>(nvec + (size_t)G * Dv);
    SmallNode* cur = reinterpret_cast<SmallNode*>(lrec + leaf_most);
    SmallNode* nxt = cur + node_most;
    SmallNode* chain = nxt + node_most;
    unsigned char* fmap = reinterpret_cast<unsigned char*>(CHAIN ? chain + node_most : chain);
    __shared__ float b_s[kMaxGroup], hp_s[kMaxGroup][3];
    __shared__ int left_s[kMaxGroup], pre_s[kMaxGroup + 1], start_s[kMaxGroup], pair_s[kMaxGroup][2];
    __shared__ int piece_s[CHAIN ? kMaxGroup + 1 : 1], lefts_s[CHAIN ? kTailMost / 64 + kMaxGroup : 1];      // pieces of 64 members before a node's, lefts of a piece
    __shared__ int n_cur_s, n_nxt_s, nrec_s, kind_s[2], base_s[2], lev_s, mx_s, mn_s, n_def_s;
    __shared__ int n_chain_s[2], chain_base_s[2], n_chain_all_s;     // (front and back of the queue)
    __shared__ int seen_s, unsure_s;        // points tested over all levels of the subtree, and left to the exact test

    const auto finish = [&](const int task) {
    if (task == 0 && threadIdx.x == 0) phase_tick(ctr, P.mid ? 3 : 2);
    const TreeNode tk = tasks[task];
    const size_t toff = (size_t)tk.tree * (size_t)P.N;
    const int* src = (tk.buf ? perm1 : perm0) + toff;
    int* dst = perm_out + toff;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    if (tk.leaf) {
        // already a bucket (any size): move it to the output buffer and record it
        if (src != dst)
            for (int i = tid; i < tk.count; i += TB) dst[tk.start + i] = src[tk.start + i] & kIdMask;
        if (tid == 0) {
            emit_leaf(tk.tree, tk.start, tk.count, tk.depth, leaf_cap, leaf_start, leaf_size, stats, ctr);
            if (recs_all) index_bucket(recs_all + (size_t)tk.tree * rec_cap, rec_cap, tk.rec, tk.start, tk.count, ctr);
        }
        return;
    }
    if (CHAIN && tk.count <= P.chain_max) {
        if (src != dst)
            for (int i = tid; i < tk.count; i += TB) dst[tk.start + i] = src[tk.start + i] & kIdMask;
        if (tid == 0) {
            const bool back = !often_in_vain(tk.count, P.MIN);
            const int at = atomicAdd(back ? &ctr->n_chain_back : &ctr->n_chain, 1);
            if (at < chain_cap) chain_all[back ? chain_cap - 1 - at : at] = tk; else ctr->overflow = 1;
        }
        return;
    }
    TreeRec* recs = recs_all ? recs_all + (size_t)tk.tree * rec_cap : nullptr;
    int* n_rec = &stats[tk.tree].n_rec;
    for (int i = tid; i < tk.count; i += TB) seg[i] = src[tk.start + i] & kIdMask;
    if (tid == 0) {
        SmallNode r;
        r.start = 0; r.count = tk.count; r.dstart = tk.dstart - tk.start; r.dcount = tk.dcount;
        r.depth = tk.depth; r.vain = 0; r.key = tk.key; r.rec = tk.rec;
        cur[0] = r;
        n_cur_s = 1; n_nxt_s = 0; nrec_s = 0; kind_s[0] = 0; kind_s[1] = 0; lev_s = 0; mx_s = 0; mn_s = 0x7fffffff;
        seen_s = 0; unsure_s = 0; n_chain_s[0] = 0; n_chain_s[1] = 0; n_chain_all_s = 0;
    }
    __syncthreads();

    auto record_leaf = [&](int start, int count, int depth, int rec) {
        if (recs) index_bucket(recs, rec_cap, rec, tk.start + start, count, ctr);
        const int at = atomicAdd(&nrec_s, 1);
        const int rank = atomicAdd(&kind_s[count > kBucketSplit ? 1 : 0], 1);
        if (at < leaf_most) lrec[at] = make_int2(tk.start + start, count | (rank << 16)); else ctr->overflow = 1;
        atomicMax(&lev_s, depth + 1);
        atomicMax(&mx_s, count);
        atomicMin(&mn_s, count);
    };

    const int grp = tid / LPP, sub = tid & (LPP - 1);       // groups of LPP lanes, one point each per iteration
    constexpr int kTailBatch = CHAIN && Q8 && KU == 1 ? 4 : 2;       // points per group and call of the screen
    while (true) {
        const int n_cur = n_cur_s;
        if (n_cur == 0) break;
        for (int b0 = 0; b0 < n_cur; b0 += G) {
            const int nb = min(G, n_cur - b0);
            // the drawn pairs of the nodes of the group, and where their points sit in the flat numbering
            if (tid < nb) {
                const SmallNode nd = cur[b0 + tid];
                int r1, r2;
                pick_pair(nd.key, nd.dcount, r1, r2);
                pair_s[tid][0] = seg[nd.dstart + r1];
                pair_s[tid][1] = seg[nd.dstart + r2];
                start_s[tid] = nd.start;
            }
            if (tid == 0) {
                n_def_s = 0;
                int run = 0;
                int pieces = 0;
                for (int j = 0; j < nb; ++j) {
                    const int count = cur[b0 + j].count;
                    pre_s[j] = run;
                    run += count;
                    if (CHAIN) {
                        piece_s[j] = pieces;
                        pieces += (count + 63) >> 6;
                    }
                }
                pre_s[nb] = run;
                if (CHAIN) piece_s[nb] = pieces;
            }
            __syncthreads();
            for (int j = wave; j < nb; j += TB / 64) {
                make_hyperplane_wave<Q8>(points + (size_t)pair_s[j][0] * P.D, points + (size_t)pair_s[j][1] * P.D, P.D,
                                         nvec + (size_t)j * Dv, hp_s[j]);
                if (lane == 0) b_s[j] = hp_s[j][0];       // written by this lane just above
            }
            for (int j = 0; j < nb; ++j) {
                const int c = pre_s[j + 1] - pre_s[j];
                for (int t = tid; t < c; t += TB) fmap[pre_s[j] + t] = (unsigned char)j;
            }
            __syncthreads();
            // side of every point of the group's nodes
            const int total = pre_s[nb];
            constexpr int kTailGroups = TB / LPP;
            const int iters = (total + kTailGroups - 1) / kTailGroups;
            for (int it = 0; it < iters; it += kTailBatch) {
                int id[kTailBatch], jj[kTailBatch], pos[kTailBatch];
                float bb[kTailBatch], h1[kTailBatch], h2[kTailBatch];
                bool valid[kTailBatch], right[kTailBatch], redo[kTailBatch];
#pragma unroll
                for (int u = 0; u < kTailBatch; ++u) {
                    const int f = (it + u) * kTailGroups + grp;
                    valid[u] = f < total;
                    jj[u] = valid[u] ? fmap[f] : 0;
                    pos[u] = valid[u] ? start_s[jj[u]] + f - pre_s[jj[u]] : 0;
                    id[u] = valid[u] ? seg[pos[u]] : 0;
                    bb[u] = b_s[jj[u]];
                    h1[u] = hp_s[jj[u]][1];
                    h2[u] = hp_s[jj[u]][2];
                }
                side_screen8<kTailBatch, Q8, LPP, KU, INSIDE>(nvec, Dv, jj, bb, h1, h2, pb16, q8, id, P.D, P.band, valid, right, redo);
#pragma unroll
                for (int u = 0; u < kTailBatch; ++u) {
                    if (valid[u] && sub == 0) {
                        if (redo[u]) tmp[atomicAdd(&n_def_s, 1)] = pos[u] | (jj[u] << 16);      // tmp is free until the partition
                        else if (right[u]) seg[pos[u]] = id[u] | (int)0x80000000;
                    }
                }
            }
            __syncthreads();
            if (tid == 0) { seen_s += total; unsure_s += n_def_s; }
            resolve_exact(TB >> 5, tid >> 5, tmp, n_def_s, nvec, Dv, b_s, points, P.D, [&](int pos) { return seg[pos] & kIdMask; },
                          [&](int pos, bool right) { if (right) seg[pos] |= (int)0x80000000; });
            __syncthreads();
            if constexpr (CHAIN) {
                // stable partition, 64 members of a node at a time by one wavefront: lefts are counted, then everyone moves
                // (seg -> tmp -> seg)
                const int n_pieces = piece_s[nb];
                auto node_of = [&](int c) { return __popcll(ballot64(lane < nb && piece_s[lane] <= c)) - 1; };
                for (int c = wave; c < n_pieces; c += TB / 64) {
                    const int j = node_of(c), i = 64 * (c - piece_s[j]) + lane;
                    const bool valid = i < pre_s[j + 1] - pre_s[j];
                    const uint64_t m = ballot64(valid && seg[valid ? start_s[j] + i : 0] >= 0);
                    if (lane == 0) lefts_s[c] = __popcll(m);
                }
                __syncthreads();
                for (int c = wave; c < n_pieces; c += TB / 64) {
                    const int j = node_of(c), first = piece_s[j], st = start_s[j], i = 64 * (c - first) + lane;
                    const bool valid = i < pre_s[j + 1] - pre_s[j];
                    const int v = valid ? seg[st + i] : 0;
                    // (a node has at most 32 pieces)
                    const int x = lane < piece_s[j + 1] - first ? lefts_s[first + lane] : 0;
                    const int a = wave_sum_i(x), before = wave_sum_i(lane < c - first ? x : 0);
                    const bool right = v < 0;
                    const int lrank = before + mask_prefix(ballot64(valid && !right));
                    if (valid) tmp[st + (right ? a + i - lrank : lrank)] = v & kIdMask;
                    if (c == first && lane == 0) left_s[j] = a;
                }
                __syncthreads();
                for (int c = wave; c < n_pieces; c += TB / 64) {
                    const int j = node_of(c), i = 64 * (c - piece_s[j]) + lane, st = start_s[j];
                    if (i < pre_s[j + 1] - pre_s[j]) seg[st + i] = tmp[st + i];
                }
            } else {
                // stable partition, one wavefront per node: seg -> tmp -> seg
                for (int j = wave; j < nb; j += TB / 64) {
                    const int st = start_s[j], cnt = pre_s[j + 1] - pre_s[j];
                    int a = 0;
                    for (int r0 = 0; r0 < cnt; r0 += 64) a += __popcll(ballot64(r0 + lane < cnt && seg[st + r0 + lane] >= 0));
                    int lbase = 0;
                    for (int r0 = 0; r0 < cnt; r0 += 64) {
                        const int i = r0 + lane;
                        const bool valid = i < cnt;
                        const int v = valid ? seg[st + i] : 0;
                        const bool right = v < 0;
                        const uint64_t m = ballot64(valid && !right);
                        const int lrank = lbase + mask_prefix(m);
                        if (valid) tmp[st + (right ? a + i - lrank : lrank)] = v & kIdMask;
                        lbase += __popcll(m);
                    }
                    wave_lds_sync();
                    for (int i = lane; i < cnt; i += 64) seg[st + i] = tmp[st + i];
                    if (lane == 0) left_s[j] = a;
                }
            }
            __syncthreads();
            // children: buckets are recorded, the others wait for the next level
            if (tid < nb) {
                const SmallNode nd = cur[b0 + tid];
                TreeNode full, c0, c1;
                full.tree = tk.tree; full.start = nd.start; full.count = nd.count; full.dstart = nd.dstart;
                full.dcount = nd.dcount; full.depth = nd.depth; full.buf = 0; full.leaf = 0; full.key = nd.key;
                const int nc = split_rules(full, left_s[tid], P.MIN, P.MAX, 0, c0, c1);
                if (recs) {
                    // (index_split; one addition for the splits of the group)
                    const uint64_t both = ballot64(nc == 2);
                    const int lead = first_lane(both);
                    int base = 0;
                    if (lane == lead) base = atomicAdd(n_rec, 2 * (int)__popcll(both));
                    base = __shfl(base, max(lead, 0), 64) + 2 * mask_prefix(both);
                    c0.rec = c1.rec = nd.rec;
                    if (nc == 2) {
                        c0.rec = base;
                        c1.rec = base + 1;
                        if (base + 2 <= rec_cap && nd.rec < rec_cap) {
                            TreeRec r;
                            r.a = pair_s[tid][0]; r.b = pair_s[tid][1]; r.c0 = c0.rec; r.c1 = c1.rec;
                            recs[nd.rec] = r;
                        } else {
                            ctr->overflow = 1;
                        }
                    }
                }
                // (many subtrees: a node leaves for the chain phase when it has been split in vain kVainMost times in a row)
                bool leaves = false;
                if constexpr (!CHAIN) {
                    const bool vain = nc == 1 && !c0.leaf && c0.depth < P.MAX_DEPTH - 1;
                    leaves = vain && nd.vain >= kVainMost - 1 && c0.count <= P.chain_max;
                    const bool front = often_in_vain(c0.count, P.MIN);
                    const uint64_t m = ballot64(leaves), mf = ballot64(leaves && front), mb = m & ~mf;
                    if (m != 0) {
                        const int lead = first_lane(m);
                        int at_f = 0, at_b = 0;
                        if (lane == lead) {
                            if (mf != 0) at_f = atomicAdd(&ctr->n_chain, (int)__popcll(mf));
                            if (mb != 0) at_b = atomicAdd(&ctr->n_chain_back, (int)__popcll(mb));
                        }
                        at_f = __shfl(at_f, lead, 64) + mask_prefix(mf);
                        at_b = __shfl(at_b, lead, 64) + mask_prefix(mb);
                        if (leaves) {
                            TreeNode c = c0;
                            c.start += tk.start;
                            c.dstart += tk.start;
                            c.buf = 0;
                            c.chunk0 = 0;
                            const int at = front ? at_f : at_b;
                            if (at < chain_cap) chain_all[front ? at : chain_cap - 1 - at] = c; else ctr->overflow = 1;
                        }
                    }
                }
                auto child = [&](const TreeNode& c) {
                    if (c.leaf || c.depth >= P.MAX_DEPTH - 1) {
                        record_leaf(c.start, c.count, c.depth, c.rec);
                    } else {
                        const bool small = CHAIN && c.count <= P.chain_max;
                        const int at = atomicAdd(small ? &n_chain_all_s : &n_nxt_s, 1);
                        if (at < node_most) {
                            SmallNode sn;
                            sn.start = c.start; sn.count = c.count; sn.dstart = c.dstart; sn.dcount = c.dcount;
                            sn.depth = c.depth;
                            sn.vain = !CHAIN && nc == 1 ? nd.vain + 1 : 0;
                            sn.key = c.key; sn.rec = c.rec;
                            if (small) sn.place = atomicAdd(&n_chain_s[often_in_vain(c.count, P.MIN) ? 0 : 1], 1);
                            (small ? chain : nxt)[at] = sn;
                        } else {
                            ctr->overflow = 1;
                        }
                    }
                };
                if (!leaves) child(c0);
                if (nc == 2) child(c1);
            }
            __syncthreads();
        }
        if (tid == 0) { n_cur_s = min(n_nxt_s, node_most); n_nxt_s = 0; }
        SmallNode* t = cur; cur = nxt; nxt = t;
        __syncthreads();
    }
    for (int i = tid; i < tk.count; i += TB) dst[tk.start + i] = seg[i];
    if (tid == 0) {
        if (CHAIN) {
            chain_base_s[0] = n_chain_s[0] ? atomicAdd(&ctr->n_chain, n_chain_s[0]) : 0;
            chain_base_s[1] = n_chain_s[1] ? atomicAdd(&ctr->n_chain_back, n_chain_s[1]) : 0;
        }
        TreeStats* st = stats + tk.tree;
        base_s[0] = kind_s[0] ? atomicAdd(&st->n_leaves, kind_s[0]) : 0;
        base_s[1] = kind_s[1] ? atomicAdd(&st->n_big, kind_s[1]) : 0;
        atomicMax(&st->levels, lev_s);
        atomicMax(&st->max_leaf, mx_s);
        atomicMin(&st->min_leaf, mn_s);
        stat_add(stat, task, 0, seen_s);
        stat_add(stat, task, 1, unsure_s);
    }
    __syncthreads();
    const int nrec = min(nrec_s, leaf_most);
    for (int i = tid; i < nrec; i += TB) {
        const int2 r = lrec[i];
        const int count = r.y & 0xffff, rank = r.y >> 16;
        store_leaf(tk.tree, r.x, count, base_s[count > kBucketSplit ? 1 : 0] + rank, leaf_cap, leaf_start, leaf_size, ctr);
    }
    for (int i = tid; CHAIN && i < min(n_chain_all_s, node_most); i += TB) {
        const SmallNode sn = chain[i];
        TreeNode c;
        c.tree = tk.tree; c.start = tk.start + sn.start; c.count = sn.count; c.dstart = tk.start + sn.dstart; c.dcount = sn.dcount;
        c.depth = sn.depth; c.buf = 0; c.leaf = 0; c.rec = sn.rec; c.chunk0 = 0; c.key = sn.key;
        const int back = often_in_vain(sn.count, P.MIN) ? 0 : 1, at = chain_base_s[back] + sn.place;
        if (at < chain_cap) chain_all[back ? chain_cap - 1 - at : at] = c; else ctr->overflow = 1;
    }
    };
    if constexpr (CHAIN) {
        // (after the middle phase only the device knows how many there are)
        const int n = P.mid ? ctr->n_tail : n_tasks;
        for (int task = blockIdx.x; task < n; task += gridDim.x) {
            __syncthreads();
            finish(task);
        }
    } else if ((int)blockIdx.x < n_tasks) {
        finish(blockIdx.x);
    }
}

// ---------------------------------------------------------------------------
// middle phase: one workgroup per node of up to mid_most points
// ---------------------------------------------------------------------------
// A wide level of a batch of few points is three launches that leave most of the device idle, about 25 us whatever the level holds,
// and a tree of 10,000 points has six of them above the nodes the tail kernel takes.  Here one workgroup of 1024 threads keeps the
// permutation of a node in LDS and splits it, and whatever of its descendants is larger than P.small, one node after the other: no launch
// and no trip of the permutation to memory in between.  A node costs the trips for the pair's rows, for the screening rows and
// for the rows of the undecided points and, beyond that, the rate at which one compute unit
// reads screening rows, which sets the largest node (tree_mid_most).  The others go to the queue of the tail kernel.
// (K-NN graph of 3,000 x 200, 10 trees 889 -> 831 us, 10,000 x 32, 4 trees 624 -> 590, one tree of 10,000 x 2 235 -> 215; 123,457 x 37, 12 trees
// and one tree of 592,523 x 20, where the wide levels above remain: the same.)
constexpr int kMidMost = 12288;          // points (LDS: 4 bytes of permutation and 2 of the list of undecided points each)
constexpr int kMidThreads = 1024, kMidPer = kMidMost / kMidThreads;
constexpr int kMidOut = 64;              // nodes for the tail kernel kept before they are given a place in its queue
constexpr int kMidNext = 2;

struct MidNode : SmallNode {
    int leaf;                             // 1: a bucket, or to be one at the depth limit; kMidNext: for the next launch
};

template <int LPP, int KU, bool INSIDE>
__global__ __launch_bounds__(kMidThreads, 4) void k_mid(const float* __restrict__ points, const uint8_t* __restrict__ q8, TreeParams P, int most,
                                                        const int* __restrict__ perm0, const int* __restrict__ perm1, int* __restrict__ perm_out,
                                                        const TreeNode* __restrict__ tasks, TreeNode* __restrict__ tail, int tail_cap, int stack_cap,
                                                        TreeStats* stats, LevelCounters* ctr, TreeRec* __restrict__ recs_all, int rec_cap,
                                                        unsigned long long* __restrict__ stat, const int* n_tasks, TreeNode* __restrict__ next,
                                                        int* n_next, int next_cap)
{
    // dynamic LDS: seg[most] | nvec[nvec_len(D)] | nodes to split [stack_cap] | nodes for the tail [kMidOut] | undecided points [most]
    extern __shared__ __align__(16) unsigned char mid_lds[];
    int* seg = reinterpret_cast<int*>(mid_lds);
    float* nvec = reinterpret_cast<float*>(seg + most);
    MidNode* stack = reinterpret_cast<MidNode*>(nvec + nvec_len(P.D));
    MidNode* out = stack + stack_cap;
    uint16_t* list = reinterpret_cast<uint16_t*>(out + kMidOut);
    constexpr int kWaves = kMidThreads / 64;
    __shared__ float hp_s[4];
    __shared__ int count_s[kMidPer * kWaves], all_s, n_def_s, n_stack_s, n_out_s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (n_tasks && (int)blockIdx.x >= *n_tasks) return;
    if (blockIdx.x == 0 && tid == 0) phase_tick(ctr, 2);
    const TreeNode tk = tasks[blockIdx.x];
    if (tk.leaf || tk.count <= P.small) {
        // (nodes beside larger ones that were split at a wide level)
        if (tid == 0) {
            const int at = atomicAdd(&ctr->n_tail, 1);
            if (at < tail_cap) tail[at] = tk; else ctr->overflow = 1;
        }
        return;
    }
    const int* src = (tk.buf ? perm1 : perm0) + (size_t)tk.tree * (size_t)P.N;
    int* dst = perm_out + (size_t)tk.tree * (size_t)P.N;
    for (int i = tid; i < tk.count; i += kMidThreads) seg[i] = src[tk.start + i] & kIdMask;
    if (tid == 0) {
        MidNode r;
        r.start = 0; r.count = tk.count; r.dstart = tk.dstart - tk.start; r.dcount = tk.dcount;
        r.depth = tk.depth; r.leaf = 0; r.key = tk.key; r.rec = tk.rec;
        stack[0] = r;
        n_stack_s = 1;
        n_out_s = 0;
    }
    __syncthreads();
    // the nodes that wait for the tail kernel, or for the next launch, get their places (all threads call)
    auto give_out = [&]() {
        const int n = n_out_s;
        if (tid < n) {
            const MidNode sn = out[tid];
            TreeNode c;
            c.tree = tk.tree; c.start = tk.start + sn.start; c.count = sn.count; c.dstart = tk.start + sn.dstart; c.dcount = sn.dcount;
            c.depth = sn.depth; c.buf = 0; c.leaf = sn.leaf; c.rec = sn.rec; c.chunk0 = 0; c.key = sn.key;
            if (sn.leaf == kMidNext) {
                c.leaf = 0;
                const int at = atomicAdd(n_next, 1);
                if (at < next_cap) next[at] = c; else ctr->overflow = 1;
            } else {
                const int at = atomicAdd(&ctr->n_tail, 1);
                if (at < tail_cap) tail[at] = c; else ctr->overflow = 1;
            }
        }
        __syncthreads();
        if (tid == 0) n_out_s = 0;
        __syncthreads();
    };
    constexpr int kGroups = kMidThreads / LPP, kBatch = KU == 1 ? 4 : 2;
    const int grp = tid / LPP, sub = tid & (LPP - 1);
    int seen = 0, unsure = 0;
    // the steps of the first workgroup stand for those of all (phase_tick)
    const bool timed = blockIdx.x == 0 && tid == 0;
    long long since = timed ? (long long)wall_clock64() : 0, ticks[3] = {0, 0, 0};
    auto step = [&](int which) {
        if (!timed) return;
        const long long now = (long long)wall_clock64();
        ticks[which] += now - since;
        since = now;
    };
    while (true) {
        const int n_stack = n_stack_s;
        if (n_stack == 0) break;
        const MidNode nd = stack[n_stack - 1];
        const int st = nd.start, cnt = nd.count;
        int r1, r2;
        pick_pair(nd.key, nd.dcount, r1, r2);
        const int p1 = seg[nd.dstart + r1], p2 = seg[nd.dstart + r2];
        if (wave == 0) make_hyperplane_wave(points + (size_t)p1 * P.D, points + (size_t)p2 * P.D, P.D, nvec, hp_s);
        if (tid == 64) n_def_s = 0;
        __syncthreads();
        step(0);
        const float b = hp_s[0], n1 = hp_s[1], sn = hp_s[2];
        for (int it = 0; it * kGroups < cnt; it += kBatch) {
            int id[kBatch], jz[kBatch], pos[kBatch];
            float bb[kBatch], h1[kBatch], h2[kBatch];
            bool valid[kBatch], right[kBatch], redo[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                const int i = (it + u) * kGroups + grp;
                valid[u] = i < cnt;
                pos[u] = st + min(i, cnt - 1);
                id[u] = seg[pos[u]] & kIdMask;
                jz[u] = 0;
                bb[u] = b;
                h1[u] = n1;
                h2[u] = sn;
            }
            side_screen8<kBatch, true, LPP, KU, INSIDE>(nvec, 0, jz, bb, h1, h2, nullptr, q8, id, P.D, P.band, valid, right, redo);
#pragma unroll
            for (int u = 0; u < kBatch; ++u) {
                if (valid[u] && sub == 0) {
                    if (redo[u]) list[atomicAdd(&n_def_s, 1)] = (uint16_t)(pos[u] - st);
                    else if (right[u]) seg[pos[u]] = id[u] | (int)0x80000000;
                }
            }
        }
        __syncthreads();
        const int n_def = n_def_s;
        seen += cnt;
        unsure += n_def;
        resolve_exact(kMidThreads / 32, tid >> 5, list, n_def, nvec, 0, hp_s, points, P.D, [&](int pos) { return seg[st + pos] & kIdMask; },
                      [&](int pos, bool right) { if (right) seg[st + pos] |= (int)0x80000000; });
        __syncthreads();
        step(1);
        // stable partition: a thread's entries are at tid, tid + 1024, ..; they wait in registers while the lefts of every 64 are counted
        int v[kMidPer];
#pragma unroll
        for (int u = 0; u < kMidPer; ++u) {
            v[u] = -1;
            if (u * kMidThreads >= cnt) continue;
            const int i = u * kMidThreads + tid;
            if (i < cnt) v[u] = seg[st + i];
            const uint64_t m = ballot64(v[u] >= 0);
            if (lane == 0) count_s[u * kWaves + wave] = __popcll(m);
        }
        __syncthreads();
        if (wave == 0) {
            // lefts before each 64, and all of them
            constexpr int kEach = (kMidPer * kWaves + 63) / 64;
            const int n = (cnt + kMidThreads - 1) / kMidThreads * kWaves;
            int x[kEach], run = 0;
#pragma unroll
            for (int k = 0; k < kEach; ++k) {
                x[k] = kEach * lane + k < n ? count_s[kEach * lane + k] : 0;
                run += x[k];
            }
            int before = wave_excl_scan_i(run);
            if (lane == 63) all_s = before + run;
#pragma unroll
            for (int k = 0; k < kEach; ++k) {
                if (kEach * lane + k < n) count_s[kEach * lane + k] = before;
                before += x[k];
            }
        }
        __syncthreads();
        const int a = all_s;
#pragma unroll
        for (int u = 0; u < kMidPer; ++u) {
            if (u * kMidThreads >= cnt) continue;
            const int i = u * kMidThreads + tid;
            const int lrank = count_s[u * kWaves + wave] + mask_prefix(ballot64(v[u] >= 0));
            if (i < cnt) seg[st + (v[u] < 0 ? a + i - lrank : lrank)] = v[u] & kIdMask;
        }
        if (tid == 0) {
            TreeNode full, c0, c1;
            full.tree = tk.tree; full.start = nd.start; full.count = nd.count; full.dstart = nd.dstart; full.dcount = nd.dcount;
            full.depth = nd.depth; full.buf = 0; full.leaf = 0; full.rec = nd.rec; full.chunk0 = 0; full.key = nd.key;
            const int nc = split_rules(full, a, P.MIN, P.MAX, 0, c0, c1);
            if (recs_all) index_split(recs_all + (size_t)tk.tree * rec_cap, &stats[tk.tree].n_rec, rec_cap, nd.rec, p1, p2, nc, c0.rec, c1.rec, ctr);
            int n_left = n_stack - 1, n_out = n_out_s;
            auto child = [&](const TreeNode& c) {
                const bool forced = c.depth >= P.MAX_DEPTH - 1, split = !c.leaf && !forced && c.count > P.small;
                MidNode x;
                x.start = c.start; x.count = c.count; x.dstart = c.dstart; x.dcount = c.dcount;
                x.depth = c.depth; x.leaf = c.leaf || forced ? 1 : 0; x.rec = c.rec; x.key = c.key;
                if (split && next) x.leaf = kMidNext;
                if (!split || next) out[n_out++] = x;
                else if (n_left < stack_cap) stack[n_left++] = x;
                else ctr->overflow = 1;
            };
            child(c0);
            if (nc == 2) child(c1);
            n_stack_s = n_left;
            n_out_s = n_out;
        }
        __syncthreads();
        if (n_out_s > kMidOut - 2) give_out();
        step(2);
    }
    for (int i = tid; i < tk.count; i += kMidThreads) dst[tk.start + i] = seg[i];
    give_out();
    if (timed) {
        for (int k = 0; k < 3; ++k) ctr->phase_ticks[k] += ticks[k];
        ctr->last_tick = (long long)wall_clock64();
    }
    if (tid == 0) {
        stat_add(stat, (int)blockIdx.x, 0, seen);
        stat_add(stat, (int)blockIdx.x, 1, unsure);
    }
}

// ---------------------------------------------------------------------------
// chain phase: small nodes, finished from the distances of their points
// ---------------------------------------------------------------------------
// A node just above the leaf limit is split again, with a pair of its larger side, until a hyperplane leaves both sides
// large enough: 200 times in a row for the unluckiest node of 20,000 x 32 points in 50 trees, 430 for 70,000 x 784 with
// buckets of 91..182.  Each of these levels needs the sides of the one before, so they are a serial chain, and in the tail
// kernel a link of it costs the whole of a level of a workgroup (17,000 and 51,000 cycles at these two inputs: the trips
// to memory for the pair's rows, the points' screening rows and the undecided points' rows).  But the points stay the
// same, and which side of the hyperplane between x1 and x2 a point x is on is whether it is nearer to x1 or to x2.  So a
// workgroup bounds the distances of all pairs of the node once, and from then on a link is two reads of LDS per point and a
// partition in registers.
//
// The distances come from the matrix cores: rows less the row of the node's first point, split into two bfloat16 numbers each
// (mfma_split.hpp), 32 dimensions at a time; the sums of 32 dimensions are added up outside the matrix cores, so that their error
// does not grow with the dimension.  They are kept as 16-bit whole numbers of one unit for the node (65534: the largest), which leaves
// LDS for four nodes of 128 points per compute unit (two as floats).
//
// When a link may decide: the exact test compares fl(n.x) with fl(b), the true n.x - b is (d2 - d1) / 2, and the two evaluations
// are off by at most 1.01 (D/32 + 8) u ||n|| (||x|| + (||x1|| + ||x2||) / 2) together, u = 2^-24 (chains of D/32 terms, five steps
// of the butterfly, the roundings of n, x1 + x2 and their product; Cauchy-Schwarz), ||n|| = sqrt(d(x1, x2)).  A distance of
// the matrix is off by at most c S (mfma_split.hpp, S = sum of the squared norms less the first point, plus the rounding of that
// subtraction) and half a unit.  With the largest norms and the largest distance of the node in the place of those of the three
// points this is one number for the node: a point's side is certain when |d2 - d1| exceeds it (70,000 x 784: 10 units, 20,000 x 32: 3).
// The others (a point in some thousands) get the exact test.  Rows that are not finite or far longer than the others (32 times
// the typical squared norm) have the mark kUnknown in the place of their distances, and get the exact test as well: one
// such row must not take the resolution from the others.
//
// Where x1 and x2 have the same coordinates the normal is zero and the exact test puts every point on the left (0 < 0, or a
// comparison with NaN).  Every point is as near to one as to the other, so that d1 and d2 decide nothing, and more than MAX
// equal rows are split until the depth limit; so nodes with a pair that may be equal have their rows compared, and the number of
// the first equal row is kept for each.  (20,000 x 32, buckets of 17..34, a tenth of the points in groups of 60
// equal rows, 10 trees: 137 ms with an exact test of every point, 34 without.)
__device__ __forceinline__ int tri_at(int i, int j, int n)
{
    const int lo = min(i, j), hi = max(i, j);
    return lo * n - ((lo * (lo + 1)) >> 1) + hi - lo - 1;
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

constexpr int kUnknown = 0xffff;         // no distance: the point gets the exact test
constexpr int kChainStep = 32;           // dimensions staged at a time
constexpr int kChainPitch = kChainStep + 8;      // 16-bit numbers per staged row: an odd number of 16-byte units

// The distances of a node of up to kChainSquare points are kept as a square matrix (a point's distances to x1 are a row of it; the
// pitch lets 32 lanes write 8 bytes each down a column without conflicts), of a larger one as its upper triangle.
constexpr int kChainSquare = 128;
__host__ __device__ inline size_t chain_matrix_entries(int n)
{
    return n <= kChainSquare ? (size_t)((n + 31) & ~31) * (size_t)(((n + 31) & ~31) + 4) : (size_t)n * (n - 1) / 2;
}
__host__ __device__ inline size_t chain_up16(size_t bytes) { return (bytes + 15) & ~(size_t)15; }
// bytes of LDS: staged rows, later the distances | norms | ids (two nodes) | undecided points | stack | buckets (two nodes) | order,
// sides, equal rows | records of the index (two nodes)
__host__ __device__ inline size_t chain_region_bytes(int n)
{
    const size_t rows = (size_t)((n + 31) & ~31) * kChainPitch * 4, matrix = chain_up16(chain_matrix_entries(n) * 2);
    return rows > matrix ? rows : matrix;
}
// A record of the index of a tree that is written once the places of the node's records are known: of the node itself (at = -1) or the
// at-th of them; so are the children of a split, c0 and c0 + 1.  A bucket has c0 = -1.
struct ChainRec {
    int at, a, b, c0;
};
__host__ __device__ inline size_t chain_lds_bytes(int n, int node_cap, bool index)
{
    return chain_region_bytes(n) + (size_t)((n + 31) & ~31) * 16 + chain_up16((size_t)node_cap * (sizeof(SmallNode) + 16)) +
           3 * chain_up16((size_t)n) + (index ? (size_t)node_cap * 4 * sizeof(ChainRec) : 0);
}

// What a distance of the matrix may be off by over S = |a|^2 + |b|^2 (rows less the first one): 3 * 2^-20 S for the products that are
// dropped and what two halves leave of a number (split2_half); 32 exact products in a row, every addition within 2^-23 of the sum of
// absolute values whatever the order or rounding mode (the sums of the other products are 2^-9 of those); in units of 2^-24 S the
// additions of the steps, the squared norms (chains of D/8 terms), four times the rounding of the subtraction of the first row, and
// the final expression.
inline float chain_gram_error(int D)
{
    return 3.2f / 1048576.0f + (float)(kChainStep + 2) / 8388608.0f + (float)(D / 8 + D / 16 + 24) / 16777216.0f;
}

// The draws of the next levels of a chain.  The key of a child follows from the key of its parent and the side alone, so
// the nodes of the next five levels are worked out side by side: lane 2 h + i holds draw i (draw_u32) of the node that
// is reached from the base by the bits of h below its leading one (h = 1: the base itself).
struct ChainDraws {
    uint64_t key;        // of the node of this lane
    uint32_t draw;
    int h;               // the present node (uniform)

    __device__ __forceinline__ void start(uint64_t base)
    {
        const int lane = lane_id(), node = lane >> 1;
        key = base;
        const int depth = node > 0 ? 31 - __clz(node) : 0;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            if (s < depth) key = child_key(key, (node >> (depth - 1 - s)) & 1);
        draw = draw_u32(key, (uint32_t)(lane & 1));
        h = 1;
    }
    __device__ __forceinline__ uint64_t node_key() const
    {
        return (uint64_t)(uint32_t)read_lane_i((int)(uint32_t)key, 2 * h) |
               ((uint64_t)(uint32_t)read_lane_i((int)(uint32_t)(key >> 32), 2 * h) << 32);
    }
    // the child on side s is the next node
    __device__ __forceinline__ void descend(int s)
    {
        if (h >= 16) start(child_key(node_key(), s));
        else h = 2 * h + s;
    }
    // pick_pair of the present node.  inverse: floor((2^32 - 1) / count); the quotient it gives is at most two too small
    __device__ __forceinline__ void pair(int count, uint32_t inverse, int& r1, int& r2) const
    {
        uint32_t r = draw - __umulhi(draw, inverse) * (uint32_t)count;
        r = min(r, r - (uint32_t)count);
        r = min(r, r - (uint32_t)count);
        r1 = read_lane_i((int)r, 2 * h);
        r2 = read_lane_i((int)r, 2 * h + 1);
        if (r1 == r2) pick_pair(node_key(), count, r1, r2);
    }
};

// The exact test (resolve_exact) of n points of a chain against the hyperplane of the points i1 and i2, by one wavefront: the
// hyperplane is made again beside the products (make_hyperplane_wave: the same order), so that the rows of the pair and of the points
// are one trip to memory.
template <typename IdAt, typename Apply>
__device__ __forceinline__ void chain_exact(const float* __restrict__ points, int D, int i1, int i2, const int* list, int n, IdAt id_at, Apply apply)
{
    const int hl = lane_id() & 31, h = lane_id() >> 5;
    const float* x1 = points + (size_t)i1 * (size_t)D;
    const float* x2 = points + (size_t)i2 * (size_t)D;
    for (int base = 0; base < n; base += 4) {
        const int ia = base + h, ib = base + 2 + h;
        const bool va = ia < n, vb = ib < n;
        const int ea = list[va ? ia : 0], eb = list[vb ? ib : 0];
        const float* xa = points + (size_t)id_at(ea) * (size_t)D;
        const float* xb = points + (size_t)id_at(eb) * (size_t)D;
        float s = 0.0f, sa = 0.0f, sb = 0.0f;
        for (int d0 = hl; d0 < D; d0 += 256) {
            float t1[8], t2[8], xv[8], yv[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int d = d0 + 32 * k;
                t1[k] = d < D ? x1[d] : 0.0f;
                t2[k] = d < D ? x2[d] : 0.0f;
                xv[k] = va && d < D ? xa[d] : 0.0f;
                yv[k] = vb && d < D ? xb[d] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (d0 + 32 * k < D) {
                    const float nd = t1[k] - t2[k];
                    const float prod = nd * (t1[k] + t2[k]);
                    s = s + prod * 0.5f;
                    sa = __builtin_fmaf(nd, xv[k], sa);
                    sb = __builtin_fmaf(nd, yv[k], sb);
                }
            }
        }
        s = half_butterfly_sum(s);
        sa = half_butterfly_sum(sa);
        sb = half_butterfly_sum(sb);
        if (hl == 0) {
            if (va) apply(ea, sa < s);
            if (vb) apply(eb, sb < s);
        }
    }
}

// NT: tiles of 32 points a node may have (up to 4: distances as a square matrix).  WAVES: wavefronts that make the matrix; the
// chain is the first one's, and meanwhile the others fetch the next node's ids.
template <int NT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, NT >= 4 ? 2 : 3) void k_chain(const float* __restrict__ points, const uint8_t* __restrict__ q8,
                                               TreeParams P, float gram_error,
                                               int* __restrict__ perm_out, const TreeNode* __restrict__ tasks, int task_cap,
                                               int node_cap, int leaf_cap, int* __restrict__ leaf_start,
                                               int* __restrict__ leaf_size, TreeStats* stats, LevelCounters* ctr,
                                               TreeRec* __restrict__ recs_all, int rec_cap,
                                               unsigned long long* __restrict__ stat)
{
    extern __shared__ __align__(16) unsigned char chain_lds[];
    constexpr bool kSquare = 32 * NT <= kChainSquare;
    constexpr int kThreads = 64 * WAVES, kPitch = 32 * NT + 4;
    const int nmax = P.chain_max, npad = (nmax + 31) & ~31;
    uint16_t* stage_hi = reinterpret_cast<uint16_t*>(chain_lds);
    uint16_t* stage_lo = stage_hi + npad * kChainPitch;
    uint16_t* mat = stage_hi;                                                 // once the products are there
    float* norm = reinterpret_cast<float*>(chain_lds + chain_region_bytes(nmax));
    int* ids_all = reinterpret_cast<int*>(norm + npad);                       // of this node and of the next one
    int* tmp = ids_all + 2 * npad;
    SmallNode* stack = reinterpret_cast<SmallNode*>(tmp + npad);
    int2* lrec_all = reinterpret_cast<int2*>(stack + node_cap);               // buckets of this node and of the one before
    unsigned char* ord = reinterpret_cast<unsigned char*>(stack) + chain_up16((size_t)node_cap * (sizeof(SmallNode) + 16));      // position in the node -> place in ids
    unsigned char* mark = ord + chain_up16((size_t)nmax);                     // by position: the exact test said right
    unsigned char* same = mark + chain_up16((size_t)nmax);                    // by place: first place with the same coordinates
    ChainRec* crec_all = reinterpret_cast<ChainRec*>(same + chain_up16((size_t)nmax));
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    __shared__ float most_s[WAVES], least_s[WAVES];
    __shared__ TreeNode task_s[2];
    // The queue: first the nodes that may take long (the launch lasts as long as its longest chain), then the others, in kRegions
    // regions taken in turn, so that the nodes under way belong to different trees and add to different counters.
    constexpr int kRegions = 64;
    const int n_front = ctr->n_chain, n_back = ctr->n_chain_back, region = (n_back + kRegions - 1) / kRegions;
    const int n_tasks = n_front + region * kRegions;
    const bool vec_ok = (P.D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) & 15) == 0);
    const float u24 = 1.0f / 16777216.0f;
    int seen = 0, unsure = 0;
    constexpr int kV = (NT + 1) / 2;                                          // points per lane
    uint32_t inverse[kV];                                                     // lane l: of l + 1, l + 65, ..
#pragma unroll
    for (int v = 0; v < kV; ++v) inverse[v] = 0xffffffffu / (uint32_t)((threadIdx.x & 63) + 1 + 64 * v);
    // buckets and records of the node before that have not been stored yet: their places are being reserved
    int pend_n = 0, pend_recs = 0, pend_tree = 0, pend_rec = 0, pend_base[3] = {0, 0, 0};
    auto store_pending = [&](int which, int lane) {
        const int2* lrec = lrec_all + which * node_cap;
        const int b0 = __builtin_amdgcn_readfirstlane(pend_base[0]), b1 = __builtin_amdgcn_readfirstlane(pend_base[1]);
        for (int i = lane; i < min(pend_n, node_cap); i += 64) {
            const int2 r = lrec[i];
            const int m = r.y & 0xffff, rank = r.y >> 16;
            store_leaf(pend_tree, r.x, m, (m > kBucketSplit ? b1 : b0) + rank, leaf_cap, leaf_start, leaf_size, ctr);
        }
        if (recs_all) {
            const ChainRec* crec = crec_all + which * 2 * node_cap;
            const int base = __builtin_amdgcn_readfirstlane(pend_base[2]);
            for (int i = lane; i < min(pend_recs, 2 * node_cap); i += 64) {
                const ChainRec c = crec[i];
                const int at = c.at < 0 ? pend_rec : base + c.at;
                TreeRec r;
                r.a = c.a; r.b = c.b;
                r.c0 = c.c0 < 0 ? -1 : base + c.c0;
                r.c1 = c.c0 < 0 ? -1 : base + c.c0 + 1;
                if (max(at, r.c1) < rec_cap) recs_all[(size_t)pend_tree * rec_cap + at] = r; else ctr->overflow = 1;
            }
        }
        pend_n = 0;
    };

    // (the nodes before gridDim.x of a share are the first ones of its workgroups)
    auto take_next = [&]() {
        constexpr int S = LevelCounters::kShares;
        const int mine = (int)blockIdx.x % S;
        return mine + S * (((int)gridDim.x - mine + S - 1) / S + atomicAdd(&ctr->share[mine].taken, 1));
    };
    int turn = 0, next = blockIdx.x;                                          // (next: in the fetching wavefront)
    constexpr int kFetcher = WAVES > 1 ? 1 : 0;
    while (true) {
        // (what follows from the thread's number is worked out for each node: kept across the chain it costs registers)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63;
        int* ids = ids_all + turn * npad;
        int2* lrec = lrec_all + turn * node_cap;
        if (wave == kFetcher) {
            int task = __builtin_amdgcn_readfirstlane(next), place = task;
            while (task >= n_front && task < n_tasks) {
                const int i = (task - n_front) % kRegions * region + (task - n_front) / kRegions;
                place = task_cap - 1 - i;
                if (i < n_back) break;
                int again = 0;
                if (lane == 0) again = take_next();                           // (the last region has no such node)
                task = place = __builtin_amdgcn_readfirstlane(again);
            }
            if (task < n_tasks) {
                const TreeNode t = tasks[place];
                const int* from = perm_out + (size_t)t.tree * (size_t)P.N + t.start;
                for (int i = lane; i < t.count; i += 64) ids[i] = from[i];
                if (lane == 0) task_s[turn] = t;
            } else if (lane == 0) {
                task_s[turn].tree = -1;
            }
        }
        __syncthreads();                                                      // (and the node before is done with the LDS)
        // (everything about the node in scalar registers: the chain's state is the wavefront's, not its lanes')
        TreeNode tk = task_s[turn];
        tk.tree = uniform(tk.tree);
        if (tk.tree < 0) break;
        tk.start = uniform(tk.start); tk.dstart = uniform(tk.dstart); tk.dcount = uniform(tk.dcount); tk.depth = uniform(tk.depth);
        tk.rec = uniform(tk.rec);
        tk.key = (uint64_t)(uint32_t)uniform((int)(uint32_t)tk.key) | ((uint64_t)(uint32_t)uniform((int)(uint32_t)(tk.key >> 32)) << 32);
        const int n = uniform(tk.count), nt = (n + 31) >> 5;
        int* seg = perm_out + (size_t)tk.tree * (size_t)P.N + tk.start;
        // accumulator e of lane l in tile (ti, tj): pair (32 ti + 8 (e / 4) + e % 4 + 4 (l / 32), 32 tj + l % 32); the tiles of the
        // upper triangle, column by column, are dealt out to the wavefronts
        constexpr int kTiles = (NT * (NT + 1) / 2 + WAVES - 1) / WAVES;
        f32x16 acc[kTiles];
        int tile_i[kTiles], tile_j[kTiles];
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            int k = wave + WAVES * t, tj = 0;
            while (k > tj) { k -= tj + 1; ++tj; }
            tile_i[t] = k;
            tile_j[t] = tj;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][e] = 0.0f;
        }
        float first_norm = 0.0f;                                              // squared norm of the row that is taken off the others
        float unit;                                                           // rows are multiplied by this power of two
        {
            constexpr int kRows = kThreads / 8, kLoads = 32 * NT / kRows;     // rows per pass; eight threads have 32 dimensions of a row
            float4 pre[kLoads], base;
            float nrm[kLoads];
#pragma unroll
            for (int i = 0; i < kLoads; ++i) nrm[i] = 0.0f;
            auto request = [&](int d0) {
                const int d = d0 + 4 * (tid & 7);
                base = make_float4(0.f, 0.f, 0.f, 0.f);
                if (d < P.D) base = load_dims(points + (size_t)ids[0] * (size_t)P.D + d, P.D - d, vec_ok);
#pragma unroll
                for (int i = 0; i < kLoads; ++i) {
                    const int row = (tid >> 3) + kRows * i;
                    pre[i] = base;
                    if (row < n && d < P.D) pre[i] = load_dims(points + (size_t)ids[row] * (size_t)P.D + d, P.D - d, vec_ok);
                }
            };
            request(0);
            // the largest coordinate of the node's finite rows: from the headers of the 8-bit rows, else from the rows themselves
            float top = 0.0f;
            if (q8) {
                for (int i = tid; i < n; i += kThreads) {
                    const float4 head = *reinterpret_cast<const float4*>(q8 + (size_t)ids[i] * (size_t)q8_pitch(P.D));
                    const float m = fmaxf(fabsf(head.y), fabsf(head.y + 255.0f * head.z)) * 1.01f;
                    if (head.w < INFINITY && m < 1e37f) top = fmaxf(top, m);
                }
            } else {
                for (int i = tid >> 3; i < n; i += kRows) {
                    const float* x = points + (size_t)ids[i] * (size_t)P.D;
                    for (int d = tid & 7; d < P.D; d += 8)
                        if (fabsf(x[d]) < 1e37f) top = fmaxf(top, fabsf(x[d]));
                }
            }
            top = wave_max(top);
            if (WAVES > 1) {
                if (lane == 0) most_s[wave] = top;
                __syncthreads();
#pragma unroll
                for (int w = 0; w < WAVES; ++w) top = fmaxf(top, most_s[w]);
            }
            // differences stay below 2^15
            {
                const int e = (int)(__float_as_uint(top) >> 23);              // top < 2^(e - 126)
                unit = __uint_as_float((uint32_t)min(max(127 + 14 + 126 - e, 1), 254) << 23);
                if (!(top > 0.0f)) unit = 1.0f;
            }
            for (int d0 = 0; d0 < P.D; d0 += kChainStep) {
                base.x *= unit; base.y *= unit; base.z *= unit; base.w *= unit;
                first_norm = __builtin_fmaf(base.x, base.x, first_norm); first_norm = __builtin_fmaf(base.y, base.y, first_norm);
                first_norm = __builtin_fmaf(base.z, base.z, first_norm); first_norm = __builtin_fmaf(base.w, base.w, first_norm);
#pragma unroll
                for (int i = 0; i < kLoads; ++i) {
                    const int row = (tid >> 3) + kRows * i;
                    if (row < 32 * nt) {
                        // (the products with a power of two are exact)
                        const float x = __builtin_fmaf(pre[i].x, unit, -base.x), y = __builtin_fmaf(pre[i].y, unit, -base.y);
                        const float z = __builtin_fmaf(pre[i].z, unit, -base.z), w = __builtin_fmaf(pre[i].w, unit, -base.w);
                        uint2 h, l;
                        split2_half(x, y, h.x, l.x);
                        split2_half(z, w, h.y, l.y);
                        *reinterpret_cast<uint2*>(&stage_hi[row * kChainPitch + 4 * (tid & 7)]) = h;
                        *reinterpret_cast<uint2*>(&stage_lo[row * kChainPitch + 4 * (tid & 7)]) = l;
                        nrm[i] = __builtin_fmaf(x, x, nrm[i]); nrm[i] = __builtin_fmaf(y, y, nrm[i]);
                        nrm[i] = __builtin_fmaf(z, z, nrm[i]); nrm[i] = __builtin_fmaf(w, w, nrm[i]);
                    }
                }
                __syncthreads();
                if (d0 + kChainStep < P.D) request(d0 + kChainStep);
#pragma unroll
                for (int t = 0; t < kTiles; ++t) {
                    if (tile_j[t] >= nt) continue;
                    __builtin_amdgcn_sched_barrier(0);
                    const int ra = (32 * tile_i[t] + (lane & 31)) * kChainPitch + 8 * (lane >> 5);
                    const int rb = (32 * tile_j[t] + (lane & 31)) * kChainPitch + 8 * (lane >> 5);
                    f32x16 sum;
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[e] = 0.0f;
#pragma unroll
                    for (int k = 0; k < kChainStep; k += 16) {
                        const f16x8 ah = *reinterpret_cast<const f16x8*>(&stage_hi[ra + k]), bl = *reinterpret_cast<const f16x8*>(&stage_lo[rb + k]);
                        const f16x8 al = *reinterpret_cast<const f16x8*>(&stage_lo[ra + k]), bh = *reinterpret_cast<const f16x8*>(&stage_hi[rb + k]);
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, sum, 0, 0, 0);
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, sum, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    acc[t] += sum;
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int e = 0; e < 16; ++e) sum[e] = 0.0f;
#pragma unroll
                    for (int k = 0; k < kChainStep; k += 16) {
                        const f16x8 ah = *reinterpret_cast<const f16x8*>(&stage_hi[ra + k]), bh = *reinterpret_cast<const f16x8*>(&stage_hi[rb + k]);
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, sum, 0, 0, 0);
                    }
                    acc[t] += sum;
                }
                __syncthreads();
            }
            // the eight threads of a row add up their squares
#pragma unroll
            for (int i = 0; i < kLoads; ++i) {
                float s = nrm[i];
                s += dpp_f<kDppXor1>(s); s += dpp_f<kDppXor2>(s); s += dpp_f<kDppHalfMirror>(s);
                const int row = (tid >> 3) + kRows * i;
                if ((tid & 7) == 0 && row < 32 * nt) norm[row] = row < n && s < 1e37f ? s : INFINITY;
            }
            first_norm += dpp_f<kDppXor1>(first_norm); first_norm += dpp_f<kDppXor2>(first_norm); first_norm += dpp_f<kDppHalfMirror>(first_norm);
        }
        __syncthreads();
        // typical squared norm: the mean of the exponents (every wavefront for itself)
        float norm_most = 0.0f;
        bool wild;                                                            // there is a row without distances
        {
            int ex = 0, some = 0;
            float s[kV];
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                s[v] = lane + 64 * v < n ? norm[lane + 64 * v] : 0.0f;
                const bool counts = s[v] > 0.0f && s[v] < INFINITY;
                ex += counts ? (int)(__float_as_uint(s[v]) >> 23) : 0;
                some += __popcll(ballot64(counts));
            }
            ex = wave_sum_i(ex);
            const float norm_limit = fminf(__uint_as_float((uint32_t)min((some ? ex / some : 0) + 6, 250) << 23), 1e37f);
            bool far = false;
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                if (s[v] <= norm_limit) norm_most = fmaxf(norm_most, s[v]);
                else far = true;
            }
            norm_most = wave_max(norm_most);
            wild = ballot64(far) != 0;                                        // (all wavefronts have read the same)
            // rows without distances get an infinite norm, rows beyond the node (zeros) one that makes their distances ordinary ones;
            // every wavefront writes the same
            __syncthreads();
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                if (s[v] > norm_limit) norm[lane + 64 * v] = INFINITY;
                if (lane + 64 * v >= n && lane + 64 * v < 32 * nt) norm[lane + 64 * v] = norm_most;
            }
            wave_lds_sync();
        }
        // the products become distances (infinite, or NaN, where one of the norms is)
        const float cap = 4.1f * norm_most;                                   // above the distances that are known
        float most = 0.0f, least = INFINITY;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            if (tile_j[t] >= nt) continue;
            __builtin_amdgcn_sched_barrier(0);                                // (the norms of one tile at a time: registers)
            const float nj = norm[32 * tile_j[t] + (lane & 31)];
            const int own = (lane & 31) - 4 * (lane >> 5);                    // (a row's distance to itself, in a tile on the diagonal)
            const bool diagonal = tile_i[t] == tile_j[t];
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const float4 n4 = *reinterpret_cast<const float4*>(&norm[32 * tile_i[t] + 8 * e4 + 4 * (lane >> 5)]);
                const float ni[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    const float d = __builtin_fmaf(-2.0f, acc[t][4 * e4 + x], ni[x] + nj);
                    acc[t][4 * e4 + x] = d;
                    most = fmaxf(most, fminf(d, cap));
                    if (!diagonal || own != 8 * e4 + x) least = fminf(least, d);
                }
            }
        }
        most = wave_max(most);
        least = -wave_max(-least);
        if (lane == 0) { most_s[wave] = most; least_s[wave] = least; }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WAVES; ++w) { most = fmaxf(most, most_s[w]); least = fminf(least, least_s[w]); }
        // what a distance may be off by: of all terms, in units of the norms, and what rows lose below the least 16-bit number
        const float off_d = gram_error * 2.0f * norm_most + 4.5f / 16384.0f * __builtin_sqrtf((float)P.D * norm_most) + (float)P.D * 4e-9f;
        // (nothing is certain where all distances are tiny, or a sum of the exact test could leave the range of fp32)
        const float longest = __builtin_sqrtf(norm_most) + __builtin_sqrtf(first_norm), back = 1.0f / unit;
        const bool usable = most * back * back > 1e-28f && most * back * back < 2e37f && longest * back < 2e19f;
        const float scale = usable ? 65534.0f / most : 0.0f;
        const float off = 2.0f * off_d + 4.3f * (float)(P.D / 32 + 8) * u24 * __builtin_sqrtf(most + off_d) * longest + 1e-30f * unit * unit;
        const float off_units = off * scale + 1.04f;                          // (a distance is rounded to within half a unit)
        const int limit = uniform(usable && off_units < 60000.0f ? (int)off_units : 1 << 20);
        auto entry = [&](int i, int j) { return kSquare ? i * kPitch + j : tri_at(i, j, n); };
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
            if (tile_j[t] >= nt) continue;
            __builtin_amdgcn_sched_barrier(0);
            const int j = 32 * tile_j[t] + (lane & 31), i0 = 32 * tile_i[t] + 4 * (lane >> 5);
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                uint32_t v[4];
#pragma unroll
                for (int x = 0; x < 4; ++x)
                    v[x] = (uint32_t)__builtin_amdgcn_fmed3f(__builtin_fmaf(acc[t][4 * e4 + x], scale, 0.5f), 0.0f, (float)kUnknown + 0.5f);
                const int i = i0 + 8 * e4;
                if constexpr (kSquare) {
                    // (both triangles of a tile on the diagonal: they differ by less than the error)
                    *reinterpret_cast<uint2*>(&mat[j * kPitch + i]) = make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
#pragma unroll
                    for (int x = 0; x < 4; ++x) mat[(i + x) * kPitch + j] = (uint16_t)v[x];
                } else {
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        if (i + x < j && j < n) mat[tri_at(i + x, j, n)] = (uint16_t)v[x];
                }
            }
        }
        if (wild) {
            __syncthreads();
            for (int i = 0; i < n; ++i) {
                if (norm[i] < INFINITY) continue;
                for (int j = tid; j < n; j += kThreads) {
                    if constexpr (kSquare) { mat[i * kPitch + j] = kUnknown; mat[j * kPitch + i] = kUnknown; }
                    else if (i != j) mat[tri_at(i, j, n)] = kUnknown;
                }
            }
        }
        __syncthreads();
        const bool equal_rows = uniform(least <= off_d ? 1 : 0) != 0;
        if (equal_rows) {
            // same[j]: the first place whose row has the coordinates of row j, of up to four that are near enough (eight lanes compare)
            const int near = (int)fminf(off_d * scale + 2.0f, 65534.0f);
            for (int j = tid >> 3; j < n; j += kThreads / 8) {
                int first = j;
                for (int from = 0, tries = 0; tries < 4; ++tries) {
                    int i = j;
                    for (int c = from + (tid & 7); c < j && i == j; c += 8)
                        if (mat[entry(c, j)] <= near) i = c;
#pragma unroll
                    for (int o = 1; o < 8; o <<= 1) i = min(i, __shfl_xor(i, o, 64));
                    if (i == j) break;
                    const float* xi = points + (size_t)ids[i] * (size_t)P.D;
                    const float* xj = points + (size_t)ids[j] * (size_t)P.D;
                    int differ = 0;
                    for (int d = tid & 7; d < P.D && !differ; d += 8) differ = xi[d] == xj[d] ? 0 : 1;
#pragma unroll
                    for (int o = 1; o < 8; o <<= 1) differ |= __shfl_xor(differ, o, 64);
                    if (!differ) { first = i; break; }
                    from = i + 1;
                }
                if ((tid & 7) == 0) same[j] = (unsigned char)first;
            }
            __syncthreads();
        }
        if (wave == kFetcher && lane == 0) next = take_next();
        if (wave != 0) {                                                      // the chain is the first wavefront's
            turn ^= 1;
            continue;
        }
        if (pend_n) store_pending(turn ^ 1, lane);
        TreeStats* st = stats + tk.tree;
        const int levels_seen = *const_cast<volatile int*>(&st->levels), most_seen = *const_cast<volatile int*>(&st->max_leaf),
                  least_seen = *const_cast<volatile int*>(&st->min_leaf);
        ChainRec* crec = crec_all + turn * 2 * node_cap;
        int start = 0, count = n, dstart = tk.dstart - tk.start, dcount = tk.dcount, depth = tk.depth;
        int rec = -1, n_crec = 0, n_split = 0;                                // (ChainRec)
        ChainDraws draws;
        draws.start(tk.key);
        int sp = 0, nrec = 0, n_big = 0, levels = 0, largest = 0, smallest = 0x7fffffff;
        auto dist_to = [&](int o, int q) -> int {
            if constexpr (kSquare) return mat[o * kPitch + q];
            else return q == o ? 0 : mat[tri_at(q, o, n)];
        };
        int q[kV];                                                            // places of the node's points, by position
        auto take_order = [&]() {
#pragma unroll
            for (int v = 0; v < kV; ++v) q[v] = ord[min(start + lane + 64 * v, n - 1)];
        };
        auto place_at = [&](int pos) {
            int o = read_lane_i(q[0], pos & 63);
#pragma unroll
            for (int v = 1; v < kV; ++v)
                if ((pos >> 6) == v) o = read_lane_i(q[v], pos & 63);
            return o;
        };
#pragma unroll
        for (int v = 0; v < kV; ++v) {
            q[v] = min(lane + 64 * v, n - 1);
            if (lane + 64 * v < n) ord[lane + 64 * v] = (unsigned char)(lane + 64 * v);
        }
        wave_lds_sync();
        while (true) {
            int r1, r2;
            uint32_t inv = (uint32_t)read_lane_i((int)inverse[0], (dcount - 1) & 63);
#pragma unroll
            for (int v = 1; v < kV; ++v)
                if (((dcount - 1) >> 6) == v) inv = (uint32_t)read_lane_i((int)inverse[v], (dcount - 1) & 63);
            draws.pair(dcount, inv, r1, r2);
            const int o1 = place_at(dstart - start + r1), o2 = place_at(dstart - start + r2);
            int d1[kV], d2[kV];
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                d1[v] = dist_to(o1, q[v]);
                d2[v] = dist_to(o2, q[v]);
            }
            uint64_t left[kV], again[kV], all[kV];
            int a = 0, n_def = 0;
#pragma unroll
            for (int v = 0; v < kV; ++v) {
                const int rest = count - 64 * v;
                all[v] = rest >= 64 ? ~0ull : (rest > 0 ? (1ull << rest) - 1ull : 0ull);
                const int diff = d2[v] - d1[v];
                left[v] = ballot64(diff > limit) & all[v];
                again[v] = all[v] & ~left[v] & ~ballot64(diff < -limit);
            }
            if (wild) {
#pragma unroll
                for (int v = 0; v < kV; ++v) {
                    again[v] |= ballot64(max(d1[v], d2[v]) == kUnknown) & all[v];
                    left[v] &= ~again[v];
                }
            }
            if (equal_rows && uniform(same[o1]) == uniform(same[o2])) {
#pragma unroll
                for (int v = 0; v < kV; ++v) {
                    left[v] = all[v];
                    again[v] = 0;
                }
            }
#pragma unroll
            for (int v = 0; v < kV; ++v) n_def += __popcll(again[v]);
            seen += count;
            if (n_def > 0) {
                unsure += n_def;
                int at = 0;
#pragma unroll
                for (int v = 0; v < kV; ++v) {
                    if (lane_bit(again[v])) tmp[at + mask_prefix(again[v])] = lane + 64 * v;
                    at += __popcll(again[v]);
                }
                wave_lds_sync();
                chain_exact(points, P.D, ids[o1], ids[o2], tmp, n_def, [&](int pos) { return ids[ord[start + pos]]; },
                            [&](int pos, bool right) { mark[pos] = right ? 1 : 0; });
                wave_lds_sync();
#pragma unroll
                for (int v = 0; v < kV; ++v) {
                    const bool mine = lane_bit(again[v]);
                    left[v] |= ballot64(mine && mark[mine ? lane + 64 * v : 0] == 0);
                }
            }
#pragma unroll
            for (int v = 0; v < kV; ++v) a += __popcll(left[v]);
            const int r = count - a;
            if (a != 0 && r != 0) {
                // stable partition
                int lbase = 0;
#pragma unroll
                for (int v = 0; v < kV; ++v) {
                    const int i = lane + 64 * v;
                    const int lrank = lbase + mask_prefix(left[v]);
                    const bool is_left = lane_bit(left[v]);
                    if (i < count) ord[start + (is_left ? lrank : a + i - lrank)] = (unsigned char)q[v];
                    lbase += __popcll(left[v]);
                }
                wave_lds_sync();
            }
            // (split_rules without the nodes around it) one child that stays to be split: the next link.  (It leaves no record in
            // the index of the tree either, and takes over the one of its parent.)
            if (min(a, r) < P.MIN && count > P.MAX && depth + 1 < P.MAX_DEPTH - 1) {
                ++depth;
                if (a == 0 || r == 0) {
                    draws.descend(a ? 0 : 1);
                    dstart = start;
                    dcount = count;
                    continue;
                }
                const bool left_big = a >= r;
                draws.descend(left_big ? 0 : 1);
                dstart = left_big ? start : start + a;
                dcount = left_big ? a : r;
                take_order();
                continue;
            }
            // children (split_rules): the first one that is no bucket is next, another waits on the stack
            const uint64_t key = draws.node_key();
            const bool two = min(a, r) >= P.MIN && a != 0 && r != 0;
            int rec0 = rec;
            if (two) {
                // (index_split)
                if (recs_all) {
                    if (lane == 0 && n_crec < 2 * node_cap) {
                        ChainRec x;
                        x.at = rec; x.a = ids[o1]; x.b = ids[o2]; x.c0 = 2 * n_split;
                        crec[n_crec] = x;
                    }
                    ++n_crec;
                }
                rec0 = 2 * n_split;
                ++n_split;
            }
            ++depth;
            bool have = false;
            auto child = [&](int cstart, int ccount, int cdstart, int cdcount, int side, bool leaf, int crec_at) {
                if (leaf || depth >= P.MAX_DEPTH - 1) {
                    const bool big = ccount > kBucketSplit;
                    if (lane == 0) {
                        if (nrec < node_cap) lrec[nrec] = make_int2(tk.start + cstart, ccount | ((big ? n_big : nrec - n_big) << 16));
                        if (recs_all && n_crec < 2 * node_cap) {
                            ChainRec x;
                            x.at = crec_at; x.a = tk.start + cstart; x.b = ccount; x.c0 = -1;
                            crec[n_crec] = x;
                        }
                    }
                    ++n_crec;
                    ++nrec;
                    n_big += big ? 1 : 0;
                    levels = max(levels, depth + 1);
                    largest = max(largest, ccount);
                    smallest = min(smallest, ccount);
                } else if (!have) {
                    have = true;
                    start = cstart; count = ccount; dstart = cdstart; dcount = cdcount;
                    rec = crec_at;
                    draws.start(child_key(key, side));
                } else {
                    if (lane == 0) {
                        if (sp < node_cap) {
                            SmallNode sn;
                            sn.start = cstart; sn.count = ccount; sn.dstart = cdstart; sn.dcount = cdcount;
                            sn.depth = depth; sn.key = child_key(key, side); sn.rec = crec_at;
                            stack[sp] = sn;
                        } else {
                            ctr->overflow = 1;
                        }
                    }
                    sp = min(sp + 1, node_cap);
                }
            };
            const int start0 = start, count0 = count;
            if (two) {
                child(start0, a, start0, a, 0, a <= P.MAX - 2, rec0);
                child(start0 + a, r, start0 + a, r, 1, r <= P.MAX - 2, rec0 + 1);
            } else if (a == 0 || r == 0) {
                child(start0, count0, start0, count0, a ? 0 : 1, count0 <= P.MAX - 2, rec0);
            } else {
                const bool left_big = a >= r;
                child(start0, count0, left_big ? start0 : start0 + a, left_big ? a : r, left_big ? 0 : 1, count0 <= P.MAX, rec0);
            }
            if (!have) {
                if (sp == 0) break;
                --sp;
                wave_lds_sync();
                const SmallNode* sn = &stack[sp];
                start = uniform(sn->start);
                count = uniform(sn->count);
                dstart = uniform(sn->dstart);
                dcount = uniform(sn->dcount);
                depth = uniform(sn->depth);
                rec = uniform(sn->rec);
                draws.start((uint64_t)(uint32_t)uniform((int)(uint32_t)sn->key) | ((uint64_t)(uint32_t)uniform((int)(uint32_t)(sn->key >> 32)) << 32));
            }
            take_order();
        }
        for (int i = lane; i < n; i += 64) seg[i] = ids[ord[i]];
        // the places of the buckets and records are reserved here and taken after the next node's matrix
        pend_n = nrec;
        pend_recs = n_crec;
        pend_tree = tk.tree;
        pend_rec = tk.rec;
        if (lane == 0) {
            if (nrec > n_big) pend_base[0] = atomicAdd(&st->n_leaves, nrec - n_big);
            if (n_big) pend_base[1] = atomicAdd(&st->n_big, n_big);
            if (recs_all && n_split) pend_base[2] = atomicAdd(&st->n_rec, 2 * n_split);
            if (nrec > node_cap || n_crec > 2 * node_cap) ctr->overflow = 1;
            // (the extremes settle early: what they were when the chain began spares nearly all of the atomics)
            if (levels_seen < levels) atomicMax(&st->levels, levels);
            if (most_seen < largest) atomicMax(&st->max_leaf, largest);
            if (least_seen > smallest) atomicMin(&st->min_leaf, smallest);
        }
        turn ^= 1;
    }
    if (wave == 0 && pend_n) store_pending(turn ^ 1, threadIdx.x);
    if (threadIdx.x == 0) {
        stat_add(stat, (int)blockIdx.x, 0, seen);
        stat_add(stat, (int)blockIdx.x, 1, unsure);
    }
}

// What a batch tells the host at its end, in pinned memory.
struct BatchReport {
    int stats[64][5];                    // the first five of TreeStats
    long long phase_ticks[4];
    unsigned long long counts[2];
    int overflow;
    int seq;
};

__global__ __launch_bounds__(64) void k_tree_report(const TreeStats* __restrict__ stats, int nb, LevelCounters* ctr,
                                                    const unsigned long long* __restrict__ stat, BatchReport* out, int seq)
{
    const int lane = threadIdx.x;
    if (lane == 0) phase_tick(ctr, 3);
    if (lane < nb) {
        const TreeStats s = stats[lane];
        int* o = out->stats[lane];
        o[0] = s.n_leaves; o[1] = s.n_big; o[2] = s.levels; o[3] = s.max_leaf; o[4] = s.min_leaf;
    }
    static_assert(kStatSlots == 64, "one slot per lane");
    unsigned long long a = stat[kStatPitch * lane], b = stat[kStatPitch * lane + 1];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    if (lane < 4) out->phase_ticks[lane] = ctr->phase_ticks[lane];
    if (lane == 0) {
        out->counts[0] = a;
        out->counts[1] = b;
        out->overflow = ctr->overflow;
    }
    __threadfence_system();
    if (lane == 0) __hip_atomic_store(&out->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <typename T>
int dmalloc(T** p, size_t n)
{
    return ws_alloc(reinterpret_cast<void**>(p), std::max<size_t>(n, 1) * sizeof(T));
}

}  // namespace

// ---------------------------------------------------------------------------
// host driver
// ---------------------------------------------------------------------------
struct TreeBatchWorkspace {
    int B = 0, N = 0;
    int leaf_cap = 0, node_cap = 0, tail_cap = 0, chunk_cap = 0;
    int* perm[2] = {nullptr, nullptr};   // perm[0] is also the output
    TreeNode* nodes[2] = {nullptr, nullptr};
    TreeNode* tail = nullptr;
    TreeNode* chain = nullptr;           // nodes for the chain phase
    TreeNode* mid = nullptr;             // nodes for the middle phase (when there is one)
    int mid_most = 0;                    // points of the largest of them
    TreeNode* mid_next = nullptr;        // nodes for its second launch, and for its third: mid_next_cap each
    int mid_next_cap = 0;
    int* chunk2node = nullptr;
    int* chunk_left = nullptr;
    float* planes = nullptr;             // hyperplanes of the nodes of the current wide level: node_cap x (4 + nvec_len(D))
    uint8_t* side_ops = nullptr;         // ... and their records for the side tests by the 8-bit copy
    int* leaf_start = nullptr;
    int* leaf_size = nullptr;
    TreeStats* stats = nullptr;
    LevelCounters* ctr = nullptr;
    int D = 0;
    LevelNotes notes;                    // pinned
    BatchReport* h_report = nullptr;     // pinned
    unsigned long long* stat = nullptr;  // kStatSlots x kStatPitch: counts for the report (stat_add)
    unsigned long long counts[2] = {0, 0};       // of the last batch: points the side tests looked at, undecided ones
    // index of the trees for routing query points (allocated by tree_ws_enable_index)
    TreeRec* recs = nullptr;             // B x rec_cap
    int rec_cap = 0;
    float phase_s[4] = {0.f, 0.f, 0.f, 0.f};   // of the last batch: side tests, hyperplanes, scatter, tail kernel
    // side tests of the first levels taken point by point (tree_sweep.hpp); allocated when D allows it
    int pm_ks = 0;                       // 32-dimension steps of a row as matrix-core operands (1, 2, 4, 8), 0 = not available
    int pm_W = 0;                        // tiles of 32 points (even)
    int pm_Bs = 0;                       // B rounded up to 16
    uint8_t* pm_path = nullptr;          // 32 W x Bs
    uint32_t* pm_side = nullptr;         // B x W
    uint32_t* pm_undec = nullptr;        // B x W
    int* pm_map[2] = {nullptr, nullptr}; // B x pm::kPaths, this level's and the next one's
    pm::PlaneQ* pm_sc = nullptr;         // B x pm::kPaths
    int8_t* pm_aq = nullptr;             // B x pm::kMaxGroups x 32 x 32 pm_ks
    int2* pm_child = nullptr;            // node_cap
};

static void free_ws(TreeBatchWorkspace& w)
{
    void* dev[] = {w.perm[0], w.perm[1], w.nodes[0], w.nodes[1], w.tail, w.chain, w.mid, w.mid_next, w.chunk2node,
                   w.chunk_left, w.leaf_start, w.leaf_size, w.stats, w.ctr, w.recs, w.planes, w.side_ops,
                   w.pm_path, w.pm_side, w.pm_undec, w.pm_map[0], w.pm_map[1], w.pm_sc, w.pm_aq, w.pm_child, w.stat};
    for (void* p : dev) ws_free(p);
    pin_free(w.notes.block());
    pin_free(w.h_report);
    w = TreeBatchWorkspace();
}

void tree_ws_free(TreeBatchWorkspace* w)
{
    if (!w) return;
    free_ws(*w);
    delete w;
}

int tree_ws_leaf_cap(const TreeBatchWorkspace* w) { return w->leaf_cap; }
const int* tree_ws_perm(const TreeBatchWorkspace* w, int t) { return w->perm[0] + (size_t)t * w->N; }
const int* tree_ws_leaf_start(const TreeBatchWorkspace* w, int t) { return w->leaf_start + (size_t)t * w->leaf_cap; }
const int* tree_ws_leaf_size(const TreeBatchWorkspace* w, int t) { return w->leaf_size + (size_t)t * w->leaf_cap; }

const int* tree_ws_stats(const TreeBatchWorkspace* w, int t)
{
    return reinterpret_cast<const int*>(w->stats + t);
}

// Nodes of at most this many points are finished by one workgroup (k_tail): 1024, or 2048 for short rows, where a
// wide level costs more per byte of row it reads (the permutation entries it moves weigh more) -- measured on 10M x 32
// points 4.46 against 4.81 ms per tree, on 1M x 100 points 0.548 against 0.520 -- and for batches so small (N x B below
// 2^21 points) that the subtrees do not fill the device anyway: a wide level then costs its launches and little else
// (70,000 x 784, 10 trees: 0.964 against 0.996 ms per tree).  RSFK_TREE_SMALL overrides (tests).
int tree_small_threshold(int D, int N, int B)
{
    const char* e = std::getenv("RSFK_TREE_SMALL");
    const bool few = (size_t)N * (size_t)std::max(B, 1) < ((size_t)1 << 21);
    const int v = e && *e ? std::atoi(e) : (D <= 48 || few ? 2048 : 1024);
    return std::min(kTailMost, std::max(64, v));
}
// Largest node the chain phase takes (0: none).  Up to 128 points the matrix costs less than the two or three levels of the tail
// kernel it stands for.  Larger nodes only where they are likely to be split in vain, which means that less than a quarter of their points is more
// than the two sides need (3,000 x 200 with buckets of 31..128: one split and a half per node, tail and chains 142 -> 181 us).
int tree_chain_max(int D, int MIN, int MAX)
{
    const char* e = std::getenv("RSFK_TREE_CHAIN");
    if ((e && e[0] == '0') || D > 2048) return 0;
    if (MAX <= 40) return 64;
    if (MAX + MAX / 8 <= kChainSquare) return kChainSquare;
    const int n = std::min(256, 8 * MIN / 3);
    return n > MAX ? n : 0;
}
// Largest node the middle phase takes (0: there is none): batches of few points (tree_small_threshold), and nodes whose screening
// rows one compute unit reads in the time of a wide level, about a megabyte (12,288 points of 32 dimensions, 4,608 of 200).
// RSFK_TREE_MID=0 switches it off, =n limits the size (tests).
int tree_mid_most(int D, int N, int B, int small)
{
    if ((size_t)N * (size_t)std::max(B, 1) >= ((size_t)1 << 21)) return 0;
    int n = std::min(kMidMost, (1 << 20) / q8_pitch(D) + 512) & ~63;
    int least = small + small / 2;
    if (const char* e = std::getenv("RSFK_TREE_MID")) {
        n = std::min(n, std::atoi(e) & ~63);
        least = small + 1;
    }
    return n >= least && N > small ? n : 0;
}

// bytes of device memory a batch of B trees needs (three lists of nodes: tail, chain phase, middle phase)
size_t tree_ws_bytes(int N, int D, int MIN, int B)
{
    const size_t lc = (size_t)N / (size_t)std::max(MIN, 1) + 2;
    return bf16_copy_bytes(N, D) + (size_t)B * ((size_t)N * 8 + (size_t)N * 2 + 512 * 1024 + lc * (8 + 3 * sizeof(TreeNode)) + ((size_t)N / 1024 + 2) * (2 * sizeof(TreeNode) + 24 + (size_t)(4 + nvec_len(D)) * 4 + side_op_bytes(D)));
}

// From now on every build with this workspace also writes the index of each tree (TreeRec records).
int tree_ws_enable_index(TreeBatchWorkspace* w, int MIN, int MAX_DEPTH)
{
    if (w->recs) return 0;
    // buckets <= N / MIN + 1 and two-child nodes fewer than buckets (one-child nodes leave no record)
    (void)MAX_DEPTH;
    const size_t cap = (size_t)2 * ((size_t)w->N / (size_t)std::max(MIN, 1) + 2) + 64;
    RSFK_CHECK(cap < ((size_t)1 << 30), "tree index: too many nodes");
    w->rec_cap = (int)cap;
    if (dmalloc(&w->recs, (size_t)w->B * cap)) return 1;
    return 0;
}
const TreeRec* tree_ws_recs(const TreeBatchWorkspace* w, int t) { return w->recs + (size_t)t * w->rec_cap; }
int tree_ws_rec_cap(const TreeBatchWorkspace* w) { return w->rec_cap; }
const int* tree_ws_n_rec(const TreeBatchWorkspace* w, int t) { return &w->stats[t].n_rec; }

int tree_ws_alloc(TreeBatchWorkspace** out, int N, int D, int MIN, int B)
{
    TreeBatchWorkspace* w = new TreeBatchWorkspace();
    *out = w;
    w->B = B; w->N = N; w->D = D;
    const int small = tree_small_threshold(D, N, B);
    w->leaf_cap = N / std::max(MIN, 1) + 2;
    w->node_cap = B * (N / small + 2);
    w->tail_cap = B * w->leaf_cap;
    w->chunk_cap = B * (N / kWideChunk + N / small + 4) + 16;      // sum ceil(count/chunk) <= N/chunk + nodes
    if (dmalloc(&w->perm[0], (size_t)B * N)) return 1;
    if (dmalloc(&w->perm[1], (size_t)B * N)) return 1;
    if (dmalloc(&w->nodes[0], (size_t)w->node_cap)) return 1;
    if (dmalloc(&w->nodes[1], (size_t)w->node_cap)) return 1;
    if (dmalloc(&w->tail, (size_t)w->tail_cap)) return 1;
    if (dmalloc(&w->chain, (size_t)w->tail_cap)) return 1;
    w->mid_most = tree_mid_most(D, N, B, small);
    // (nodes above `small`, no two with a point in common, are handed on; a few kilobytes)
    w->mid_next_cap = (int)((size_t)N * (size_t)B / (size_t)(small + 1)) + 1;
    if (w->mid_most && (dmalloc(&w->mid, (size_t)w->tail_cap) || dmalloc(&w->mid_next, 2 * (size_t)w->mid_next_cap))) return 1;
    if (dmalloc(&w->chunk2node, (size_t)w->chunk_cap)) return 1;
    if (dmalloc(&w->chunk_left, (size_t)w->chunk_cap)) return 1;
    if (dmalloc(&w->planes, (size_t)w->node_cap * (size_t)(4 + nvec_len(D)))) return 1;
    if (dmalloc(&w->side_ops, (size_t)w->node_cap * side_op_bytes(D))) return 1;
    if (dmalloc(&w->leaf_start, (size_t)B * w->leaf_cap)) return 1;
    if (dmalloc(&w->leaf_size, (size_t)B * w->leaf_cap)) return 1;
    if (dmalloc(&w->stats, (size_t)B)) return 1;
    if (dmalloc(&w->ctr, (size_t)1)) return 1;
    if (dmalloc(&w->stat, (size_t)kStatSlots * kStatPitch)) return 1;
    if (D <= 256 && N > small && B <= 64) {
        w->pm_ks = D <= 32 ? 1 : D <= 64 ? 2 : D <= 128 ? 4 : 8;
        w->pm_W = 2 * ((N + 63) / 64);                     // an even number of 32-point tiles
        w->pm_Bs = (B + 15) & ~15;
        if (dmalloc(&w->pm_path, (size_t)w->pm_Bs * w->pm_W * 32)) return 1;
        if (dmalloc(&w->pm_side, (size_t)w->pm_Bs * w->pm_W)) return 1;
        if (dmalloc(&w->pm_undec, (size_t)w->pm_Bs * w->pm_W)) return 1;
        if (dmalloc(&w->pm_map[0], (size_t)B * pm::kPaths)) return 1;
        if (dmalloc(&w->pm_map[1], (size_t)B * pm::kPaths)) return 1;
        if (dmalloc(&w->pm_sc, (size_t)B * pm::kPaths)) return 1;
        if (dmalloc(&w->pm_aq, (size_t)B * pm::kMaxGroups * 32 * 32 * w->pm_ks)) return 1;
        if (dmalloc(&w->pm_child, (size_t)w->node_cap)) return 1;
    }
    void* notes = nullptr;
    if (pin_alloc(&notes, LevelNotes::kBytes)) return 1;
    if (pin_alloc(reinterpret_cast<void**>(&w->h_report), sizeof(BatchReport))) {
        pin_free(notes);
        return 1;
    }
    w->notes.set(notes, &w->h_report->seq);
    return 0;
}

// seconds the last batch spent in: side tests, hyperplanes of the wide levels, scatter, tail kernel
const float* tree_ws_phase_seconds(const TreeBatchWorkspace* w) { return w->phase_s; }
// of the last batch: [0] points the side tests of all levels and trees looked at (the sum over the levels of the
// members of the nodes that were split), [1] those the screen left to the exact fp32 test
const unsigned long long* tree_ws_counts(const TreeBatchWorkspace* w) { return w->counts; }
// bytes of a row of the copy the side tests are screened on
int tree_screen_row_bytes(int D, bool q8) { return q8 ? q8_pitch(D) : 2 * bf16_pitch(D); }

// Builds nb (<= B) trees with seeds seed0 .. seed0+nb-1.  pb16 = rows of the bfloat16 copy of the points (may be
// null: every side test then reads the fp32 row).  On return perm[0] of
// tree t holds the point ids grouped by bucket and (leaf_start, leaf_size)[t]
// the buckets, in no particular order: those of at most kBucketSplit points in entries [0, n_small), the
// larger ones in entries [leaf_cap - n_big, leaf_cap).  host_stats receives 5 ints per tree: number of
// buckets, number of levels, largest and smallest bucket, number of large buckets.
int build_tree_batch(TreeBatchWorkspace* w, const float* points, const uint16_t* pb16, const uint8_t* q8, int N, int D, int MIN, int MAX,
                     int MAX_DEPTH, int seed0, int nb, int* host_stats, hipStream_t stream)
{
    RSFK_CHECK(nb >= 1 && nb <= w->B && N == w->N && D == w->D, "tree batch: workspace does not match the request");
    RSFK_CHECK(N >= 1 && D >= 1, "tree batch: N and D must be positive");
    TreeParams P;
    P.N = N; P.D = D; P.MIN = MIN; P.MAX = MAX; P.MAX_DEPTH = MAX_DEPTH;
    P.small = tree_small_threshold(D, N, w->B);
    P.chain_max = tree_chain_max(D, MIN, MAX);
    P.chunk = kWideChunk;
    // bfloat16 rounding 2^-8 (1 + 2^-7), plus the summation errors of the screen (D/8 terms per lane and a 3-step
    // tree) and of the exact test (D/32 terms per lane and a 5-step tree), 1 % on top
    P.band = 1.01f * ((1.0f + 1.0f / 128.0f) / 256.0f + (float)(D / 8 + D / 32 + 16) / 16777216.0f);

    RSFK_CHECK(nb <= 64, "tree batch: at most 64 trees at a time");
    // Levels whose side tests are taken point by point (needs the 8-bit copy).  RSFK_PM_LEVELS overrides (0 = none).
    // The sweep multiplies every tile of points with every block of 16 hyperplanes of a tree, so its cost doubles
    // per level from the fifth on; measured, the seventh level is the last one it takes faster than k_side_q8 (with six: trees of 10M x 32 37.9 -> 38.7 ms,
    // of 1M x 256 26.4 -> 26.9), the sixth where a row is a single line and the sweep's operands are those of 128 dimensions (1M x 72, 96, 112, 25 trees:
    // 11.5, 11.6, 12.3 -> 11.2, 11.5, 12.0; 64, 120 dimensions 9.8, 15.0 -> 9.8, 15.2).  Batches of
    // less than 2^22 points do not fill the device either way, and k_side_q8 is one launch instead of four.
    int pm_levels = 0;
    if (q8 && w->pm_ks) {
        const int last = D > 64 && q8_pitch(D) == 128 ? pm::kMaxLevels - 2 : pm::kMaxLevels - 1;
        pm_levels = (size_t)N * (size_t)nb >= ((size_t)1 << 22) ? last : 0;
        if (const char* e = std::getenv("RSFK_PM_LEVELS")) pm_levels = std::max(0, std::min(pm::kMaxLevels, std::atoi(e)));
    }
    NodeQueues Q;
    Q.next = w->nodes[0]; Q.next_cap = w->node_cap; Q.chunk_cap = w->chunk_cap; Q.slot = 0;
    // The middle phase needs the 8-bit copy, and is for launches over few subtrees (below; RSFK_TAIL_BLOCK=256: as with many).
    const char* tail_block = std::getenv("RSFK_TAIL_BLOCK");
    const bool tail_q8 = q8 != nullptr && std::getenv("RSFK_TAIL_BF16") == nullptr;
    const bool mid = w->mid_most > 0 && tail_q8 && pm_levels == 0 && !(tail_block && std::atoi(tail_block) < 1024);
    P.mid = mid ? 1 : 0;
    TreeParams PW = P;                                                        // of the wide levels
    if (mid) PW.small = w->mid_most;
    Q.tail = mid ? w->mid : w->tail; Q.tail_cap = w->tail_cap;
    Q.ctr = w->ctr;
    Q.n_tail = mid ? &w->ctr->n_mid : &w->ctr->n_tail;
    w->notes.begin();
    {
        const size_t total = (size_t)N * nb;
        const int grid = (int)std::min<size_t>((total + 255) / 256, 65536);
        hipLaunchKernelGGL(k_tree_init, dim3(grid), dim3(256), 0, stream, w->perm[0], Q, PW, nb, seed0,
                           pm_levels > 0 ? w->pm_map[0] : nullptr, w->stats, w->stat);
        RSFK_HIP(hipGetLastError());
    }

    int cur = 0;
    const size_t side_lds = (size_t)(4 + nvec_len(D)) * sizeof(float);
    RSFK_CHECK(side_lds <= kSideRecordMost, "tree batch: D too large for the LDS of the side test");
    // k_level_planes: four nodes per workgroup while their records fit in 48 KB, else one
    const int plane_waves = 4 * side_lds <= 48 * 1024 ? 4 : 1;
    if (side_lds > 48 * 1024) {
        RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_level_planes), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)side_lds));
        RSFK_HIP(hipFuncSetAttribute(q8 ? reinterpret_cast<const void*>(k_side_q8<true>) : reinterpret_cast<const void*>(k_side),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)side_lds));
    }
    for (float& v : w->phase_s) v = 0.0f;
    // Wide levels.  A level is three launches over bounds on its counts, which follow from the counts of the level before:
    // the host reads those from pinned memory while the level before runs, so the stream never waits for the host (a copy
    // and a synchronisation per level took 14 us, and the table of chunks two launches more).  One level too many is
    // queued at the end; its workgroups find nothing to do.
    int n_tail = nb, level = 0;
    size_t most_nodes = (size_t)nb, most_chunks = (size_t)nb * (((size_t)N + P.chunk - 1) / P.chunk);
    while (N > PW.small) {
        if (level > 0) {
            const LevelNote* note = w->notes.of(level - 1);
            if (wait_for_word(&note->seq, LevelNotes::seq(level - 1), stream)) return 1;
            RSFK_CHECK(!note->overflow && note->n_nodes <= w->node_cap && note->n_chunks <= w->chunk_cap,
                       "tree batch: node queue overflow");
            n_tail = note->n_tail;
            if (std::getenv("RSFK_TREE_TRACE"))
                std::fprintf(stderr, "level %d: %d nodes, %d chunks, tail %d\n", level - 1, note->n_nodes, note->n_chunks, note->n_tail);
            if (note->n_nodes == 0) break;
            // a split makes two nodes of one and adds at most one chunk
            most_nodes = std::min<size_t>(2 * (size_t)note->n_nodes, (size_t)w->node_cap);
            most_chunks = std::min<size_t>((size_t)note->n_chunks + (size_t)note->n_nodes, (size_t)w->chunk_cap);
        }
        const int slot = level & 3;
        const int n_chunks = (int)std::min<size_t>(most_chunks, (size_t)w->chunk_cap);
        int* ctr_chunks = &w->ctr->queue[slot].chunks;
        const bool swept = level < pm_levels;
        hipLaunchKernelGGL(k_level_planes, dim3((unsigned)((most_nodes + plane_waves - 1) / plane_waves)), dim3(64 * plane_waves),
                           plane_waves * side_lds, stream, points, PW, w->perm[0], w->perm[1], w->nodes[cur], level, w->node_cap,
                           w->planes, q8 && !swept ? w->side_ops : nullptr, w->chunk2node, w->ctr, w->stat, w->notes.of(level),
                           LevelNotes::seq(level));
        if (swept) {
            // the sides of every point in all trees of the batch, then their marks in the permutations
            const int n_paths = 1 << level, ks = w->pm_ks, W = w->pm_W;
            const int rec = 4 + nvec_len(D);
            hipLaunchKernelGGL(pm::k_pm_planes, dim3((unsigned)((nb * n_paths + 3) / 4)), dim3(256), 0, stream, w->planes, rec, D,
                               32 * ks, w->pm_map[level & 1], n_paths, nb, w->pm_sc, w->pm_aq);
            const dim3 sgrid((unsigned)((W + 7) / 8));          // two tiles per wavefront, four wavefronts
#define RSFK_SWEEP_LAUNCH(KS)                                                                                                \
            hipLaunchKernelGGL((pm::k_pm_sweep<KS>), sgrid, dim3(256), 0, stream, q8, N, D, nb, w->pm_Bs, level, W, w->pm_path, \
                               w->pm_side, w->pm_undec, w->pm_aq, w->pm_sc)
            if (ks == 1) RSFK_SWEEP_LAUNCH(1);
            else if (ks == 2) RSFK_SWEEP_LAUNCH(2);
            else if (ks == 4) RSFK_SWEEP_LAUNCH(4);
            else RSFK_SWEEP_LAUNCH(8);
#undef RSFK_SWEEP_LAUNCH
            const size_t words = (size_t)nb * W;
            hipLaunchKernelGGL(pm::k_pm_resolve, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream, points, D, W,
                               w->pm_Bs, words, w->pm_path, w->pm_sc, w->planes, rec, w->pm_side, w->pm_undec, w->stat);
            hipLaunchKernelGGL(k_pm_mark, dim3(n_chunks), dim3(kBlock), 0, stream, P, w->perm[0], w->perm[1], w->nodes[cur],
                               ctr_chunks, w->chunk2node, w->chunk_left, w->pm_side, W);
        } else {
#define RSFK_SIDE_LAUNCH(LINE)                                                                                                 \
            hipLaunchKernelGGL(k_side_q8<LINE>, dim3(n_chunks), dim3(kBlock), side_lds, stream, points, q8, P, w->perm[0], w->perm[1], \
                               w->nodes[cur], slot, w->ctr, w->chunk2node, w->chunk_left, w->planes, w->side_ops, w->stat)
            if (!q8)
                hipLaunchKernelGGL(k_side, dim3(n_chunks), dim3(kBlock), side_lds, stream, points, pb16, P, w->perm[0], w->perm[1],
                                   w->nodes[cur], slot, w->ctr, w->chunk2node, w->chunk_left, w->planes, w->stat);
            else if (q8_pitch(D) == 64) RSFK_SIDE_LAUNCH(false);
            else RSFK_SIDE_LAUNCH(true);
#undef RSFK_SIDE_LAUNCH
        }
        const bool map_next = level + 1 < pm_levels;
        Q.next = w->nodes[cur ^ 1];
        Q.slot = (level + 1) & 3;
        hipLaunchKernelGGL(k_scatter, dim3(n_chunks), dim3(kBlock), 0, stream, PW, w->perm[0], w->perm[1], w->nodes[cur],
                           slot, w->chunk2node, w->chunk_left, Q, w->recs, w->stats, w->rec_cap,
                           map_next ? w->pm_child : nullptr);
        if (map_next) {
            const int n_paths = 1 << level;
            hipLaunchKernelGGL(pm::k_pm_next_map, dim3((unsigned)((nb * n_paths + 255) / 256)), dim3(256), 0, stream,
                               w->pm_map[level & 1], w->pm_map[(level + 1) & 1], w->pm_child, n_paths, nb);
        }
        RSFK_HIP(hipGetLastError());
        cur ^= 1;
        ++level;
    }
    // tail
    // Few subtrees (small inputs, few trees): what counts is how long the longest of them takes.  Workgroups of 1024 threads
    // while every subtree has a compute unit to itself, of 512 beyond that (so that all of them are resident at once:
    // 20,000 x 32, 50 trees, 808 subtrees 1.69 -> 1.58 ms for the trees), and every node the chain phase takes leaves for it.
    // With more subtrees than that the device is full anyway and that would only add the matrices (1M x 100, 50 trees: tail 10.9 ->
    // 9.5 ms, chains 9.9 ms), so a node stays until it has been split in vain kVainMost times in a row: those that
    // never come to an end keep a workgroup waiting for one node, a level per split.  Whole build without / with, kVainMost = 4:
    // clustered points 82,121 x 244, K = 5, 50 trees 32.3 -> 15.0 ms; 200,000 x 100, K = 8, 40 trees 29.6 -> 13.2; 1M x 16, K = 4, 20 trees
    // 48.0 -> 32.1; 1M x 256, K = 32, 20 trees 93.5 -> 91.5; uniform points 1M x 100, K = 32, 50 trees 51.7 -> 50.3; 1M x 32, K = 5, 10 trees
    // 11.37 -> 11.46.  After 1, 2 or 3 splits in vain the last three take 94.6 / 93.6 / 93.4, 52.0 / 50.7 / 50.3, 12.9 / 12.2 / 11.9 ms.
    // RSFK_TAIL_BLOCK=256 / 1024: as with many / as with few subtrees, whatever their number.
    RSFK_CHECK(n_tail <= w->tail_cap, "tree batch: tail queue overflow");
    if (mid && n_tail > 0) {
        const int stack_cap = w->mid_most / std::max(P.small, 1) + 4;
        const size_t lds = (size_t)w->mid_most * 6 + (size_t)nvec_len(D) * 4 + (size_t)(stack_cap + kMidOut) * sizeof(MidNode);
        const int pieces = q8_padded(D) / 16;
        // A workgroup splits one node after the other, about 10 us each; where several of its descendants will be larger than P.small, a launch ends
        // with the children, which the next one takes side by side.  A launch more is about 10 us too, so not below four times P.small, but of
        // one or two nodes from three times on (there into two launches).  Calls of trees alone, one launch -> with the children handed on: one tree of 4,300 x 2
        // 243 -> 247 us, 5,000 x 20 263 -> 267, 6,500 x 100 359 -> 338, 8,100 x 20 307 -> 299, 12,000 x 2 324 -> 311, 18,500 x 20 403 -> 385; four trees of 5,000 x 32
        // 235 -> 244, 8,000 x 4 278 -> 286, 12,000 x 4 322 -> 301; 2 to 50 trees of 7,000 points 0.95 to 1.03 (mean 1.00), of 8,500 to 22,000 0.94 to 1.05 (0.985).
        // Not with many nodes, when those of the last launch wait for each other's compute units: 20,000 x 32, 50 trees 111 -> 125 us.
        const int largest = std::min(N, w->mid_most);
        int hand = 0;
        if (n_tail <= 64 && largest > 4 * P.small) hand = 2;
        else if (n_tail <= 2 && largest > 3 * P.small) hand = 1;
        for (int pass = 0; pass <= hand; ++pass) {
            const TreeNode* tasks = pass == 0 ? w->mid : w->mid_next + (size_t)(pass - 1) * (size_t)w->mid_next_cap;
            const int* n_tasks = pass == 0 ? nullptr : &w->ctr->n_mid_next[pass - 1];
            TreeNode* next = pass == hand ? nullptr : w->mid_next + (size_t)pass * (size_t)w->mid_next_cap;
            // (nodes above P.small, no two with a point in common; two at most from each of the launch before)
            const unsigned grid = pass == 0 ? (unsigned)n_tail
                                            : (unsigned)std::max<size_t>(1, std::min((size_t)n_tail << pass, (size_t)N * (size_t)nb / (size_t)(P.small + 1)));
#define RSFK_MID_LAUNCH(L, U)                                                                                               \
            do {                                                                                                           \
                auto* kernel = header_inside<L>(D) ? k_mid<L, U, true> : k_mid<L, U, false>;                                   \
                RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
                hipLaunchKernelGGL(kernel, dim3(grid), dim3(kMidThreads), lds, stream, points, q8, P, w->mid_most, w->perm[0], w->perm[1], \
                                   w->perm[0], tasks, w->tail, w->tail_cap, stack_cap, w->stats, w->ctr, w->recs, w->rec_cap, w->stat, n_tasks, \
                                   next, pass < hand ? &w->ctr->n_mid_next[pass] : nullptr, w->mid_next_cap);                   \
            } while (0)
            if (pieces <= 2) RSFK_MID_LAUNCH(2, 1);
            else if (pieces <= 4) RSFK_MID_LAUNCH(4, 1);
            else if (pieces <= 16) RSFK_MID_LAUNCH(4, 4);
            else RSFK_MID_LAUNCH(8, 4);
#undef RSFK_MID_LAUNCH
            RSFK_HIP(hipGetLastError());
        }
        // (how many nodes it leaves to the tail only the device knows; that many are usual, and the tail kernel takes any number)
        n_tail = (int)std::min<size_t>((size_t)N * (size_t)nb * 5 / (size_t)(3 * P.small) + (size_t)nb, (size_t)w->tail_cap);
    }
    bool few = n_tail > 0 && n_tail < 8 * 256;
    if (tail_block) few = std::atoi(tail_block) >= 1024;
    if (mid) few = true;
    if (n_tail > 0) {
        // (the tail kernel keeps the bfloat16 screen: measured, it is not faster with the 8-bit one)
        // buckets of a subtree: at most small / MIN + 1; nodes of a level that are no buckets, and those for the chain phase: MAX - 1 points
        // or more each (split_rules), no two with a point in common.  Hyperplanes kept together: as many as 24 KB hold, at most kMaxGroup, and
        // fewer where short buckets leave less
        constexpr size_t kTailLds = 156 * 1024;           // (the kernel's own arrays: 1 KB)
        const int leaf_most = P.small / std::max(MIN, 1) + 4, node_most = P.small / std::max({MIN, MAX - 1, 1}) + 4;
        const size_t besides = (size_t)(2 * P.small) * 4 + (size_t)leaf_most * sizeof(int2) +
                               (few ? 3 : 2) * (size_t)node_most * sizeof(SmallNode) + (size_t)P.small;
        const size_t plane = (size_t)nvec_len(D) * 4;
        RSFK_CHECK(besides + plane <= kTailLds, "tree batch: D too large for the tail kernel's LDS budget");
        const int G = std::max(1, std::min(kMaxGroup, (int)(std::min<size_t>(24 * 1024, kTailLds - besides) / plane)));
        const size_t lds = besides + (size_t)G * plane;
#define RSFK_TAIL_LAUNCH(Q, T, C, L, U)                                                                                       \
        do {                                                                                                               \
            constexpr bool two = (L) == 2;                                                                                   \
            auto* kernel = two && header_inside<L>(D) ? k_tail<Q, T, C, L, U, two> : k_tail<Q, T, C, L, U, false>;              \
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
            hipLaunchKernelGGL(kernel, dim3(n_tail), dim3(T), lds, stream, points, pb16, q8, P, w->perm[0], w->perm[1], w->perm[0],  \
                               w->tail, n_tail, leaf_most, node_most, G, w->leaf_cap, w->leaf_start, w->leaf_size, w->stats, w->ctr, \
                               w->recs, w->rec_cap, w->stat, w->chain, w->tail_cap);                                          \
        } while (0)
        // Lanes per point: as many as there are pieces of 16 coordinates, up to four; few subtrees wait for the loads of a point, and
        // four lanes with four pieces in flight each take longer rows (eight beyond 256 dimensions).  With many subtrees eight lanes keep the
        // kernel in its registers.  (Tail of 10M x 32, 10 trees 9.25 -> 7.29 ms with two lanes instead of eight; 20,000 x 32, 50 trees
        // 306 -> 211 us, with the partition by pieces.)
        const int pieces = q8_padded(D) / 16;
#define RSFK_TAIL_LANES(T)                                                                                                  \
        do {                                                                                                               \
            if (pieces <= 2) RSFK_TAIL_LAUNCH(true, T, true, 2, 1);                                                         \
            else if (pieces <= 4) RSFK_TAIL_LAUNCH(true, T, true, 4, 1);                                                    \
            else if (pieces <= 16) RSFK_TAIL_LAUNCH(true, T, true, 4, 4);                                                   \
            else RSFK_TAIL_LAUNCH(true, T, true, 8, 4);                                                                     \
        } while (0)
        if (tail_q8 && few && n_tail <= 256) RSFK_TAIL_LANES(1024);
        else if (tail_q8 && few && (n_tail <= 512 || pieces > 4)) RSFK_TAIL_LANES(512);
        else if (tail_q8 && few) RSFK_TAIL_LANES(256);
        else if (tail_q8 && pieces <= 2) RSFK_TAIL_LAUNCH(true, 256, false, 2, 1);
        else if (tail_q8 && pieces <= 4) RSFK_TAIL_LAUNCH(true, 256, false, 4, 1);
        else if (tail_q8) RSFK_TAIL_LAUNCH(true, 256, false, 8, 1);
        else if (few) RSFK_TAIL_LAUNCH(false, 512, true, 8, 1);
        else RSFK_TAIL_LAUNCH(false, 256, false, 8, 1);
#undef RSFK_TAIL_LANES
#undef RSFK_TAIL_LAUNCH
        RSFK_HIP(hipGetLastError());
    }
    if (P.chain_max > 0) {
        const int node_cap = P.chain_max / std::max(MIN, 1) + 4;
        const size_t lds = chain_lds_bytes(P.chain_max, node_cap, w->recs != nullptr);
        const size_t most = (size_t)N * (size_t)nb / (size_t)std::max(MAX - 1, 1) + (size_t)nb;      // nodes that are no buckets are disjoint
        const unsigned grid = (unsigned)std::min<size_t>(most, 256 * (size_t)std::max<size_t>(1, (size_t)160 * 1024 / lds));
        const float gram_error = chain_gram_error(D);
#define RSFK_CHAIN_LAUNCH(NT, W)                                                                                            \
        do {                                                                                                               \
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_chain<NT, W>),                                    \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                          \
            hipLaunchKernelGGL((k_chain<NT, W>), dim3(grid), dim3(64 * W), lds, stream, points, q8, P, gram_error,           \
                               w->perm[0], w->chain, w->tail_cap, node_cap, w->leaf_cap, w->leaf_start, w->leaf_size, w->stats, w->ctr,  \
                               w->recs, w->rec_cap, w->stat);                                                               \
        } while (0)
        if (P.chain_max <= 64) RSFK_CHAIN_LAUNCH(2, 1);
        else if (P.chain_max <= kChainSquare) RSFK_CHAIN_LAUNCH(4, 2);
        else RSFK_CHAIN_LAUNCH(8, 4);
#undef RSFK_CHAIN_LAUNCH
        RSFK_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(k_tree_report, dim3(1), dim3(64), 0, stream, w->stats, nb, w->ctr, w->stat, w->h_report, LevelNotes::kReport);
    RSFK_HIP(hipGetLastError());
    if (wait_for_word(&w->h_report->seq, LevelNotes::kReport, stream)) return 1;
    const BatchReport& R = *w->h_report;
    w->counts[0] = R.counts[0];
    w->counts[1] = R.counts[1];
    {
        // the steps, from the device's clock (events between the kernels of a level would cost more than some of the
        // kernels)
        int dev = 0, khz = 0;
        if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) == hipSuccess &&
            khz > 0) {
            const float s_per_tick = 1e-3f / (float)khz;
            w->phase_s[1] = (float)R.phase_ticks[0] * s_per_tick;       // hyperplanes
            w->phase_s[0] = (float)R.phase_ticks[1] * s_per_tick;       // side tests
            w->phase_s[2] = (float)R.phase_ticks[2] * s_per_tick;       // scatter
            w->phase_s[3] = (float)R.phase_ticks[3] * s_per_tick;       // tail
        }
    }
    RSFK_CHECK(!R.overflow, "tree batch: queue overflow in the tail phase");
    for (int t = 0; t < nb; ++t) {
        const int* st = R.stats[t];
        const int total = st[0] + st[1];
        host_stats[5 * t + 0] = total;
        host_stats[5 * t + 1] = st[2];
        host_stats[5 * t + 2] = st[3];
        host_stats[5 * t + 3] = total ? st[4] : 0;
        host_stats[5 * t + 4] = st[1];
        RSFK_CHECK(total <= w->leaf_cap, "tree batch: leaf table overflow");
    }
    return 0;
}

}  // namespace rsfk
