// Query-set search, trees one after the other: the first seven levels of all trees of a batch in one kernel, on the matrix cores.
//
// Every query passes the same few nodes at the top of a tree, and k_route (ann.hip) reads their hyperplanes again for every query and
// tree: ten vector instructions per query, level and eight dimensions.  Here a wavefront keeps 64 queries as matrix-core operands and
// walks the trees: the 127 hyperplanes of a tree's first seven levels are four operand blocks of 32 (padded), a block against the queries
// is one chain of v_mfma_f32_32x32x16_f16 per 32 of them, and what is left per hyperplane and query are three instructions that turn the
// result into two bits, side and certain.  A query then walks down the bits, seven levels or to the first test that is not certain, and
// start[] says where k_route goes on.  (1M queries, 50 trees of 1M x 100: 1.8 ms for seven levels, 4.5e8 vector instructions, where
// k_route_low spends 6; the queries stay in registers for all trees of a batch, so it is bound by those instructions.)
//
// (What is certain: SideBound, ann.hpp, with the largest |b~| of the tree.)  A bucket is a node whose test is never certain: the query
// stops there.
#include "forest.hpp"
#include "ann.hpp"
#include "join_copy.hpp"
#include "wave64.hpp"
#include <algorithm>
#include <cstdlib>

namespace rsfk {

namespace {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kTopLevels = 7;
constexpr int kTopSlots = 1 << kTopLevels;        // one of them unused
constexpr int kTopBlocks = kTopSlots / 32;

// Of a tree: nodes in heap order (children of s: 2 s + 1, 2 s + 2), those of the last level and the slots below it.
struct TopTree {
    int rec[2 * kTopSlots];               // record of a slot, -1: none
    float minus_b[kTopBlocks][2][16];     // -b~ in the order of the accumulators
    uint32_t never[kTopBlocks];           // slots whose test is never certain
    float most_b;                         // largest |b~|
    int pad[3];
};

// The row of an operand block in which slot p of 32 stands, such that accumulator i of a lane of half h is slot 16 h + i.
__device__ __forceinline__ int block_row(int p) { return 8 * ((p & 15) >> 2) + 4 * (p >> 4) + (p & 3); }

// One wavefront per tree.
__global__ __launch_bounds__(64) void k_top_slots(const TreeRec* __restrict__ recs_all, const int* __restrict__ n_rec_p, int rec_cap,
                                                  TopTree* __restrict__ top_all)
{
    const int j = blockIdx.x, lane = threadIdx.x;
    const TreeRec* recs = recs_all + (size_t)j * (size_t)rec_cap;
    TopTree& top = top_all[j];
    const int n_rec = min(n_rec_p[kTreeStatPitch * j], rec_cap);
    __shared__ int rec[2 * kTopSlots];
    for (int s = lane; s < 2 * kTopSlots; s += 64) rec[s] = s == 0 && n_rec > 0 ? 0 : -1;
    if (lane < kTopBlocks) top.never[lane] = 0u;
    if (lane == 0) top.most_b = 0.0f;
    __syncthreads();
    for (int l = 0; l < kTopLevels; ++l) {
        const int s = (1 << l) - 1 + lane;
        if (lane < (1 << l) && rec[s] >= 0) {
            const TreeRec r = recs[rec[s]];
            if (r.c0 >= 0 && r.c0 < n_rec && r.c1 >= 0 && r.c1 < n_rec) {
                rec[2 * s + 1] = r.c0;
                rec[2 * s + 2] = r.c1;
            }
        }
        __syncthreads();
    }
    for (int s = lane; s < 2 * kTopSlots; s += 64) top.rec[s] = rec[s];
}

// One wavefront per slot (blockIdx.y: the tree): operand row and -b~ (normal and offset as in k_planes, ann.hip).
__global__ __launch_bounds__(256) void k_top_planes(const float* __restrict__ points, int D, const TreeRec* __restrict__ recs_all,
                                                    int rec_cap, TopTree* __restrict__ top_all, uint16_t* __restrict__ operands, int ksteps,
                                                    const float* __restrict__ mu, const float* __restrict__ scale)
{
    const int lane = threadIdx.x & 63, s = blockIdx.x * 4 + (threadIdx.x >> 6), j = blockIdx.y;
    TopTree& top = top_all[j];
    const int blk = s >> 5, p = s & 31, m = block_row(p);
    uint16_t* out = operands + ((size_t)j * kTopBlocks + blk) * (size_t)ksteps * 512 + (size_t)m * 8;
    const int rec = s < kTopSlots - 1 ? top.rec[s] : -1;
    const bool node = rec >= 0 && top.rec[2 * s + 1] >= 0;               // (a bucket has no children)
    const TreeRec r = recs_all[(size_t)j * (size_t)rec_cap + (size_t)max(rec, 0)];
    const float* x1 = points + (size_t)(node ? r.a : 0) * (size_t)D;
    const float* x2 = points + (size_t)(node ? r.b : 0) * (size_t)D;
    float b = 0.0f;
    if (lane < 32) {
        for (int d = lane; d < D; d += 32) {
            const float t1 = x1[d], t2 = x2[d];
            const float prod = (t1 - t2) * (t1 + t2);
            b = b + prod * 0.5f;
        }
    }
    b = half_butterfly_sum(b);
    b = __shfl(b, 0, 64);
    RoundedPlane pl = rounded_plane(x1, x2, D, b, mu, *scale);
    pl.sound = pl.sound && node;
    for (int d = lane; d < 16 * ksteps; d += 64)
        out[(size_t)(d >> 4) * 512 + (size_t)((d >> 3) & 1) * 256 + (d & 7)] = rounded_value(d < D ? x1[d] - x2[d] : 0.0f, pl);
    if (lane == 0) {
        top.minus_b[blk][p >> 4][p & 15] = pl.sound ? -pl.b : 0.0f;
        if (pl.sound) atomicMax(reinterpret_cast<uint32_t*>(&top.most_b), __float_as_uint(fabsf(pl.b)));
        else atomicOr(&top.never[blk], 1u << p);
    }
}

// 64 queries per wavefront, trees blockIdx.y, + gridDim.y, ...
template <int KS>
__global__ __launch_bounds__(256) void k_route_top(JoinCopy jc, int NQ, int n_trees, const TopTree* __restrict__ top_all,
                                                   const uint16_t* __restrict__ operands, const float* __restrict__ scale,
                                                   const float* __restrict__ mu_len, SideBound sb, int* __restrict__ start)
{
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    const int q0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 64;
    if (q0 >= NQ) return;                                                // the whole wavefront leaves
    const int pitch = join_pitch(jc.D);
    f16x8 x[2][KS];
    float Z[2];
    uint32_t bad[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int q = min(q0 + 32 * t + n, NQ - 1);
        const uint16_t* row = jc.rows + (size_t)q * (size_t)pitch + 8 * h;
#pragma unroll
        for (int u = 0; u < KS; ++u) x[t][u] = *reinterpret_cast<const f16x8*>(row + 16 * u);
        Z[t] = sb.query(jc.norms[q], jc.errs[q], *scale, *mu_len);
        bad[t] = Z[t] < INFINITY ? 0u : 0xffff0000u;
        if (bad[t]) Z[t] = 0.0f;
    }
    for (int j = blockIdx.y; j < n_trees; j += gridDim.y) {
        const TopTree& top = top_all[j];
        const float zb = sb.of_offset() * top.most_b;
        uint32_t side[kTopBlocks], open[kTopBlocks];                     // by slot: below the offset; not certain
#pragma unroll
        for (int blk = 0; blk < kTopBlocks; ++blk) {
            const uint16_t* op = operands + ((size_t)j * kTopBlocks + blk) * (size_t)(KS * 512) + (size_t)lane * 8;
            f32x16 a0, a1;
#pragma unroll
            for (int i = 0; i < 16; i += 4) {
                const float4 c = *reinterpret_cast<const float4*>(&top.minus_b[blk][h][i]);
                a0[i] = c.x; a0[i + 1] = c.y; a0[i + 2] = c.z; a0[i + 3] = c.w;
            }
            a1 = a0;
#pragma unroll
            for (int u = 0; u < KS; ++u) {
                const f16x8 a = *reinterpret_cast<const f16x8*>(op + u * 512);
                a0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, x[0][u], a0, 0, 0, 0);
                a1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, x[1][u], a1, 0, 0, 0);
            }
            uint32_t v[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const float z = Z[t] + zb;
                uint32_t below = 0u, unsure = 0u;
#pragma unroll
                for (int i = 15; i >= 0; --i) {
                    const float a = t == 0 ? a0[i] : a1[i];
                    below = __builtin_amdgcn_alignbit(below, __float_as_uint(a), 31);                    // << 1 | sign
                    unsure = __builtin_amdgcn_alignbit(unsure, __float_as_uint(fabsf(a) - z), 31);
                }
                v[t] = (below & 0xffffu) | (unsure << 16) | bad[t];
            }
            // lane l of the lower half: query l of the first 32, of the upper half: of the second; [0] slots 0..15, [1] slots 16..31
            const auto r = __builtin_amdgcn_permlane32_swap(v[0], v[1], false, false);
            side[blk] = (r[0] & 0xffffu) | (r[1] << 16);
            open[blk] = (r[0] >> 16) | (r[1] & 0xffff0000u) | top.never[blk];
            __builtin_amdgcn_sched_barrier(0);                           // (one block after the other: registers)
        }
        int slot = 0;
        bool go = true;
#pragma unroll
        for (int l = 0; l < kTopLevels; ++l) {
            uint32_t sw = side[0], ow = open[0];
            if (l >= 5) { const bool up = slot >= 32; sw = up ? side[1] : sw; ow = up ? open[1] : ow; }
            if (l >= 6) {
                const bool up2 = slot >= 64, up3 = slot >= 96;
                sw = up3 ? side[3] : (up2 ? side[2] : sw);
                ow = up3 ? open[3] : (up2 ? open[2] : ow);
            }
            const int at = slot & 31;
            go = go && ((ow >> at) & 1u) == 0u;
            slot = go ? 2 * slot + 1 + (int)((sw >> at) & 1u) : slot;
        }
        if (q0 + lane < NQ) start[(size_t)j * (size_t)NQ + q0 + lane] = max(top.rec[slot], 0);
    }
}

}  // namespace

// 20 trees, all levels by k_route or k_route_low -> the first seven here: 300,000 / 300,000 x 8 7.82 -> 7.67 ms, x 100 12.6 -> 12.4; 60,000
// points, 1M queries x 8 15.4 -> 14.7, x 128 26.1 -> 25.6; 20,000 / 100,000 x 50 3.21 -> 3.18; 1M / 100,000 x 8 to x 128 the same, and so are 50,000
// queries and fewer.  Few trees do not pay for the copy of the queries (ann_copy_pays).  RSFK_ANN_TOP=1 / 0 says yes or no.
bool ann_top_wanted(int n_trees, int NQ, int D)
{
    const char* e = std::getenv("RSFK_ANN_TOP");
    if (e && e[0] == '0') return false;
    if (D > 128) return false;
    if (e && e[0] == '1') return true;
    return NQ >= 100000 && ann_copy_pays(n_trees, NQ);
}

size_t ann_top_bytes(int n_trees, int D)
{
    const int ksteps = (D + 15) / 16;
    return (size_t)n_trees * (sizeof(TopTree) + (size_t)kTopBlocks * ksteps * 1024);
}

// start[j NQ + q] = the record from which query q goes on in tree j (recs, n_rec_dev as in launch_ann_forest).  jc: the copy of the
// queries.  ws: ann_top_bytes.
int launch_ann_top(const float* points, const JoinCopy& jc, int NQ, int D, int n_trees, const TreeRec* recs, const int* n_rec_dev, int rec_cap,
                   void* ws, int* start, hipStream_t stream)
{
    RSFK_CHECK(D >= 1 && D <= 128 && n_trees >= 1, "query-set search: dimensions out of range");
    const int ksteps = (D + 15) / 16;
    TopTree* top = static_cast<TopTree*>(ws);
    uint16_t* operands = reinterpret_cast<uint16_t*>(top + n_trees);
    static_assert(sizeof(TopTree) % 16 == 0, "16-byte loads");
    hipLaunchKernelGGL(k_top_slots, dim3((unsigned)n_trees), dim3(64), 0, stream, recs, n_rec_dev, rec_cap, top);
    hipLaunchKernelGGL(k_top_planes, dim3(kTopSlots / 4, (unsigned)n_trees), dim3(256), 0, stream, points, D, recs, rec_cap, top, operands,
                       ksteps, jc.mu, jc.scale());
    const unsigned gx = (unsigned)((NQ + 255) / 256);
    // (few queries: the trees are shared among more wavefronts)
    const unsigned gy = (unsigned)std::max(1, std::min(n_trees, (int)(4096 / std::max(1u, gx))));
#define RSFK_TOP(KSV)                                                                                                       \
    hipLaunchKernelGGL(k_route_top<KSV>, dim3(gx, gy), dim3(256), 0, stream, jc, NQ, n_trees, top, operands, jc.scale(), jc.mu_len(), SideBound(D), start)
    switch (ksteps) {
    case 1: RSFK_TOP(1); break;
    case 2: RSFK_TOP(2); break;
    case 3: RSFK_TOP(3); break;
    case 4: RSFK_TOP(4); break;
    case 5: RSFK_TOP(5); break;
    case 6: RSFK_TOP(6); break;
    case 7: RSFK_TOP(7); break;
    default: RSFK_TOP(8); break;
    }
#undef RSFK_TOP
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
