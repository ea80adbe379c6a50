// Bucket step of the query-set search with the pairs bounded on the matrix cores first: same results as k_ann_leaf (ann.hip),
// which evaluates every pair of a query and a member of its bucket -- nearly all of its arithmetic, though after a few trees
// hardly a pair still enters a row.
//
// A wavefront takes up to 32 queries of a bucket and the bucket 64 members at a time:
//   1. the fp32 rows are read straight into matrix-core operands, every value split into two bfloat16 numbers
//      (mfma_split.hpp); two 32 x 32 quadrants of inner products, and the squared norms;
//   2. a pair is dropped iff the lower bound of its distance, (d~ - c S)(1 - gamma) as in bucket_knn_screen.hip, is above
//      the last slot of the query's row.  NaN or infinite intermediate values never drop a pair.  A lane's accumulators are
//      the pairs of one query (members are the rows of the product, queries its columns);
//   3. the pairs that are left go to a list in LDS (room for all of them), query by query; a lane runs the sequential chain
//      of "its" pair from the two rows in the caches (the arithmetic of k_ann_leaf);
//   4. the pairs whose distance is not above the last slot are merged into the rows, four rows in flight.
// Bound by the latency of the gathers at four wavefronts per SIMD (128 registers): 1M queries / 1M x 100, the last of 50
// trees 0.57 ms where k_ann_leaf takes 0.85 (vector ALUs); the first trees, where most pairs are left, 2.9 against 1.9.  Tried: the
// members' rows of step 3 through a transposing tile in LDS (faster at D = 256 while many pairs are left, 0.65 ms here), K-NN
// rows requested before the chains run (no change), two steps of 16 dimensions in flight in separate buffers (spills).
// (Late trees of large inputs of 97 to 128 dimensions: ann_screen_half.hip, where there is room for copies of the rows.)
// No barrier: the wavefronts of a workgroup share nothing but the cache lines of a bucket they may both work on.
#include "forest.hpp"
#include "ann.hpp"
#include "exact_batch.hpp"
#include "mfma_split.hpp"
#include <algorithm>

namespace rsfk {

namespace {

constexpr int kMembers = 64;

struct alignas(16) AnnScreenLds {          // of a wavefront
    float nrm[kMembers];
    float tau[kAnnScreen];
    int qid[kAnnScreen];
    int cid[kMembers];
    uint16_t list[kAnnScreen * kMembers];  // query | member << 5
};

template <bool VEC>
__global__ __launch_bounds__(256, 4) void k_ann_screen(const float* __restrict__ points, const float* __restrict__ queries, int D, int K,
                                                    const int* __restrict__ perm, const int4* __restrict__ blk_desc,
                                                    const int* __restrict__ n_blocks, const int* __restrict__ qlist,
                                                    int* __restrict__ q_idx, float* __restrict__ q_dist, float c_err,
                                                    float one_minus_gamma, AnnForm form)
{
    if (!form.screened() || form.by_copies()) return;
    __shared__ AnnScreenLds lds_s[4];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int half = lane >> 5, r = lane & 31;
    AnnScreenLds& L = lds_s[wave];
    const int n_items = *n_blocks;
    for (int item = (int)blockIdx.x * 4 + wave; item < n_items; item += (int)gridDim.x * 4) {
        const int4 desc = blk_desc[item];
        const int start = desc.x, S = desc.y, nq = desc.w;
        const int my_q = qlist[desc.z + (r < nq ? r : 0)];                  // slots beyond nq repeat the first query
        if (half == 0) {
            L.qid[r] = my_q;
            L.tau[r] = q_dist[(size_t)my_q * (size_t)K + (size_t)(K - 1)];
        }
        const float* qp = queries + (size_t)my_q * (size_t)D;
        int n_listed = 0;
        for (int c0 = 0; c0 < S; c0 += kMembers) {
            const int nc = min(kMembers, S - c0);
            const bool two = nc > 32;
            const int my_c = perm[start + c0 + (lane < nc ? lane : 0)];
            L.cid[lane] = my_c;
            const float* p0 = points + (size_t)__shfl(my_c, r, 64) * (size_t)D;
            const float* p1 = points + (size_t)__shfl(my_c, 32 + r, 64) * (size_t)D;
            // ---- 1. two steps of 16 dimensions at a time
            f32x16 g0, g1;
#pragma unroll
            for (int i = 0; i < 16; ++i) { g0[i] = 0.0f; g1[i] = 0.0f; }
            float nrm_q = 0.0f, nrm_0 = 0.0f, nrm_1 = 0.0f;
            for (int d0 = 0; d0 < D; d0 += 32) {
                float4 a[4], b[4], c[4];
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const int d = d0 + 16 * k + 8 * half + 4 * x;
                        a[2 * k + x] = load_piece(qp, d, D, VEC);
                        b[2 * k + x] = load_piece(p0, d, D, VEC);
                        if (two) c[2 * k + x] = load_piece(p1, d, D, VEC);
                    }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    bf16x8 ah, al, bh, bl;
                    split8(a[2 * k], a[2 * k + 1], ah, al, nrm_q);
                    split8(b[2 * k], b[2 * k + 1], bh, bl, nrm_0);
                    g0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, ah, g0, 0, 0, 0);
                    g0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bl, ah, g0, 0, 0, 0);
                    g0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, al, g0, 0, 0, 0);
                    if (two) {
                        split8(c[2 * k], c[2 * k + 1], bh, bl, nrm_1);
                        g1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, ah, g1, 0, 0, 0);
                        g1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bl, ah, g1, 0, 0, 0);
                        g1 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, al, g1, 0, 0, 0);
                    }
                }
            }
            // a lane holds the squares of half of the dimensions of its row
            nrm_q += __shfl_xor(nrm_q, 32, 64);
            nrm_0 += __shfl_xor(nrm_0, 32, 64);
            nrm_1 += __shfl_xor(nrm_1, 32, 64);
            if (half == 0) {
                L.nrm[r] = nrm_0;
                L.nrm[32 + r] = nrm_1;
            }
            wave_lds_sync();
            // ---- 2. accumulator i of lane l: member 8 (i / 4) + i % 4 + 4 (l / 32) of the block, query l % 32
            const float tau = L.tau[r];
            auto screen = [&](const f32x16& g, int n0) {
                uint32_t left = 0;
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const int n = n0 + 8 * i4 + 4 * half;
                    const float4 nn4 = *reinterpret_cast<const float4*>(&L.nrm[n]);
                    const float nn[4] = {nn4.x, nn4.y, nn4.z, nn4.w};
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const float sum = nrm_q + nn[x];
                        const float dt = __builtin_fmaf(-2.0f, g[4 * i4 + x], sum);
                        const float lower = (dt - __builtin_fmaf(c_err, sum, 1e-35f)) * one_minus_gamma;
                        if (n + x < nc && !(lower > tau)) left |= 1u << (4 * i4 + x);
                    }
                }
                return r < nq ? left : 0u;
            };
            uint32_t left = screen(g0, 0) | (two ? screen(g1, 32) << 16 : 0u);
            // the pairs of query r: those of lane r, then those of lane r + 32
            const int mine = __popc(left), other = __shfl_xor(mine, 32, 64);
            const int before = wave_excl_scan_i(half == 0 ? mine + other : 0);
            int at = __shfl(before, r, 64) + (half == 0 ? 0 : other);
            const int total = read_lane_i(before, 32);
            n_listed += total;
            while (left) {
                const int i = __ffs(left) - 1;
                left &= left - 1;
                const int n = 2 * (i & ~15) + 8 * ((i & 15) >> 2) + (i & 3) + 4 * half;
                L.list[at++] = (uint16_t)(r | (n << 5));
            }
            wave_lds_sync();
            for (int off = 0; off < total; off += 64) {
                // ---- 3.
                const bool in = off + lane < total;
                const int e = in ? L.list[off + lane] : 0;
                const int m = e & 31, id = L.cid[e >> 5];
                const float* x = queries + (size_t)L.qid[m] * (size_t)D;
                const float* y = points + (size_t)id * (size_t)D;
                float acc = 0.0f;
                for (int d0 = 0; d0 < D; d0 += 32) {
                    float4 xv[8], yv[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        xv[i] = load_piece(x, d0 + 4 * i, D, VEC);
                        yv[i] = load_piece(y, d0 + 4 * i, D, VEC);
                    }
#pragma unroll
                    for (int i = 0; i < 8; ++i) {          // (zeros beyond D on both sides change nothing)
                        float df;
                        df = yv[i].x - xv[i].x; acc = __builtin_fmaf(df, df, acc);
                        df = yv[i].y - xv[i].y; acc = __builtin_fmaf(df, df, acc);
                        df = yv[i].z - xv[i].z; acc = __builtin_fmaf(df, df, acc);
                        df = yv[i].w - xv[i].w; acc = __builtin_fmaf(df, df, acc);
                    }
                }
                // ---- 4.
                const bool cand = in && acc <= L.tau[m];
                uint64_t todo = ballot64(cand);
                struct Next { int m; int ri; float rd; };
                auto next_row = [&](Next& t) {
                    t.m = -1;
                    t.ri = -2;
                    t.rd = INFINITY;
                    if (todo == 0) return;
                    t.m = read_lane_i(m, first_lane(todo));
                    todo &= ~ballot64(m == t.m);
                    if (lane < K) {
                        const size_t slot = (size_t)L.qid[t.m] * (size_t)K + (size_t)lane;
                        t.ri = q_idx[slot];
                        t.rd = q_dist[slot];
                    }
                };
                constexpr int kRows = 4;
                Next cur[kRows], nxt[kRows];
#pragma unroll
                for (int u = 0; u < kRows; ++u) next_row(cur[u]);
                while (cur[0].m >= 0) {
#pragma unroll
                    for (int u = 0; u < kRows; ++u) next_row(nxt[u]);
#pragma unroll
                    for (int u = 0; u < kRows; ++u) {
                        if (cur[u].m < 0) break;
                        KnnRow<1> row;
                        row.idx[0] = cur[u].ri;
                        row.dist[0] = cur[u].rd;
                        row.init_sorted(K);
                        row.merge(cand && m == cur[u].m, id, acc);
                        if (row.changed) {
                            const size_t slot = (size_t)L.qid[cur[u].m] * (size_t)K;
                            row.store(q_idx + slot, q_dist + slot);
                            if (lane == 0) L.tau[cur[u].m] = row.tau;
                        }
                    }
#pragma unroll
                    for (int u = 0; u < kRows; ++u) cur[u] = nxt[u];
                }
                wave_lds_sync();
            }
            wave_lds_sync();                               // done with cid, nrm and the list
        }
        if (form.counts(item) && lane == 0)
            atomicAdd(form.word(item), ((unsigned long long)((unsigned)nq * (unsigned)S) << 32) | (unsigned)n_listed);
    }
}

}  // namespace

int launch_ann_screen(const float* points, const float* queries, int D, int K, const int* perm, const int4* blk_desc,
                      const int* n_blocks, int most_blocks, const int* qlist, int* q_idx, float* q_dist, const AnnForm& form,
                      hipStream_t stream)
{
    RSFK_CHECK(K >= 1 && K <= 64, "query-set search: screened form takes K up to 64");
    const float c_err = split_gram_error_coefficient((D + 15) & ~15);
    const float one_minus_gamma = 1.0f - (float)(D + 8) * (1.0f / 4194304.0f);
    RSFK_CHECK(one_minus_gamma > 0.5f, "query-set search: D too large for the screened form");
    const unsigned grid = (unsigned)std::min(2048, (most_blocks + 3) / 4);
    const bool vec = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) | reinterpret_cast<uintptr_t>(queries)) & 15) == 0;
    if (vec)
        hipLaunchKernelGGL(k_ann_screen<true>, dim3(grid), dim3(256), 0, stream, points, queries, D, K, perm, blk_desc, n_blocks, qlist,
                           q_idx, q_dist, c_err, one_minus_gamma, form);
    else
        hipLaunchKernelGGL(k_ann_screen<false>, dim3(grid), dim3(256), 0, stream, points, queries, D, K, perm, blk_desc, n_blocks, qlist,
                           q_idx, q_dist, c_err, one_minus_gamma, form);
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
