// The screened bucket step of the query-set search (ann_screen.hip) for late trees over many rows of 97 to 128 dimensions, by float16 copies of the
// queries and the points (join_copy.hpp, the same mu and s for both): same results.
//
// In ann_screen.hip a lane reads "its" fp32 row 16 bytes at a time: a load touches up to 64 rows, comes back to a cache line seven times
// while the line is still on its way, and rows of 400 bytes straddle lines, so that the address units are busy 82 % of the time and
// 17.4 million lines are fetched where the rows are 8.2 million (1M queries / 1M x 100, the last of 50 trees).  Here a row is two lines,
// eight lanes read one together, straight into LDS:
//   1. 64 members and 32 queries, a line of each at a time, then matrix-core operands from the tile;
//   2. a pair is dropped iff |x~|^2 + |y~|^2 - 2 x~.y~, less what the sums may be off by, is above (s r + e_x + e_y)^2: r the root of the query's last
//      slot and what the fp32 chain may be below the distance, e what the rounding of a row took at most (join_err_rel, join_err_abs).  Rows that
//      are not finite never drop a pair;
//   3. the pairs that are left wait until there are 64 of them, over several items: rows of the queries, then of the members, 128 bytes at a
//      time through the tile; a lane runs the sequential chain of its pair;
//   4. the pairs whose distance is not above the last slot (as it was when the pair was listed) are merged into the rows.
// Bound by the lines it fetches: the last of 50 trees 0.565 -> 0.42 ms (14 million lines, 4.3 TB/s).  Where rows are shorter or aligned to lines the
// form above is the faster one (300,000 / 500,000, 30 trees of K = 32, ann_screen.hip -> here for all screened trees: x 80 19.7 -> 20.4, x 64 17.1
// -> 17.7, x 40 15.7 -> 17.1), and so it is in early trees and where the rows stay in the last cache (ann_half_share_q16).  One wavefront per workgroup, 11 of them per compute unit (LDS);
// 16,384 workgroups at most: 8,192 end with a tail (28.2), one item each leaves the waiting list half empty (27.1).
#include "forest.hpp"
#include "ann.hpp"
#include "exact_batch.hpp"
#include "join_bounds.hpp"
#include <algorithm>
#include <cstdlib>

namespace rsfk {

namespace {

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int kMembers = 64;
constexpr int kSteps = 8;                  // of 16 dimensions: rows of join_pitch(D) = 128 values
constexpr int kFlush = 64;                 // pairs that are evaluated together

struct alignas(16) AnnHalfLds {
    u32x4 tile[(kMembers + kAnnScreen) * 8];   // 128 bytes of a row, members then queries; piece p of row r stands at 8 r + (p ^ r % 8)
    float nrm[kMembers];
    int cid[kMembers];
    int qid[kAnnScreen];
    float tau[kAnnScreen];
    int pend_q[2 * kFlush], pend_c[2 * kFlush];      // pairs that wait: query, member, and the last slot of the query's row when listed
    float pend_tau[2 * kFlush];
};
__device__ __forceinline__ int tile_at(int row, int piece) { return 8 * row + (piece ^ (row & 7)); }

// The first n <= 64 pairs that wait: their distances, and those not above the last slot into the rows.
__device__ __forceinline__ void evaluate(AnnHalfLds& L, int n, const float* __restrict__ points, const float* __restrict__ queries, int D, int K,
                                         bool vec, int* __restrict__ q_idx, float* __restrict__ q_dist)
{
    const int lane = lane_id(), sub = lane & 7, grp = lane >> 3;
    // ---- 3. eight lanes read 128 bytes of a row; a lane gets the pieces of its pair from the tile
    const bool in = lane < n;
    const int at = in ? lane : 0;
    const int q = L.pend_q[at], id = L.pend_c[at];
    float acc = 0.0f;
    for (int d0 = 0; d0 < D; d0 += 32) {
        f32x4 xv[8];
        u32x4 xr[8], yr[8];
        const int d = d0 + 4 * sub;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int e = 8 * i + grp;
            if (e < n) {
                xr[i] = __builtin_bit_cast(u32x4, load_piece(queries + (size_t)L.pend_q[e] * (size_t)D, d, D, vec));
                yr[i] = __builtin_bit_cast(u32x4, load_piece(points + (size_t)L.pend_c[e] * (size_t)D, d, D, vec));
            }
        }
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 8; ++i) L.tile[tile_at(8 * i + grp, sub)] = xr[i];
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = __builtin_bit_cast(f32x4, L.tile[tile_at(lane, i)]);
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 8; ++i) L.tile[tile_at(8 * i + grp, sub)] = yr[i];
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < 8; ++i) {          // (zeros beyond D on both sides change nothing)
            const f32x4 y = __builtin_bit_cast(f32x4, L.tile[tile_at(lane, i)]);
            float df;
            df = y.x - xv[i].x; acc = __builtin_fmaf(df, df, acc);
            df = y.y - xv[i].y; acc = __builtin_fmaf(df, df, acc);
            df = y.z - xv[i].z; acc = __builtin_fmaf(df, df, acc);
            df = y.w - xv[i].w; acc = __builtin_fmaf(df, df, acc);
        }
    }
    // ---- 4.
    const bool cand = in && acc <= L.pend_tau[at];
    uint64_t todo = ballot64(cand);
    struct Next { int q; int ri; float rd; };
    auto next_row = [&](Next& t) {
        t.q = -1;
        t.ri = -2;
        t.rd = INFINITY;
        if (todo == 0) return;
        t.q = read_lane_i(q, first_lane(todo));
        todo &= ~ballot64(q == t.q);
        if (lane < K) {
            const size_t slot = (size_t)t.q * (size_t)K + (size_t)lane;
            t.ri = q_idx[slot];
            t.rd = q_dist[slot];
        }
    };
    constexpr int kRows = 4;
    Next cur[kRows], nxt[kRows];
#pragma unroll
    for (int u = 0; u < kRows; ++u) next_row(cur[u]);
    while (cur[0].q >= 0) {
#pragma unroll
        for (int u = 0; u < kRows; ++u) next_row(nxt[u]);
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            if (cur[u].q < 0) break;
            KnnRow<1> row;
            row.idx[0] = cur[u].ri;
            row.dist[0] = cur[u].rd;
            row.init_sorted(K);
            row.merge(cand && q == cur[u].q, id, acc);
            if (row.changed) {
                const size_t slot = (size_t)cur[u].q * (size_t)K;
                row.store(q_idx + slot, q_dist + slot);
            }
        }
#pragma unroll
        for (int u = 0; u < kRows; ++u) cur[u] = nxt[u];
    }
}

__global__ __launch_bounds__(64, 3) void k_ann_screen_half(JoinCopy qc, JoinCopy pc, const float* __restrict__ points, const float* __restrict__ queries,
                                                       int D, int K, bool vec, const int* __restrict__ perm, const int4* __restrict__ blk_desc,
                                                       const int* __restrict__ n_blocks, const int* __restrict__ qlist,
                                                       int* __restrict__ q_idx, float* __restrict__ q_dist, const float* __restrict__ scale, float kappa,
                                                       float err_rel, float err_abs, float one_minus_gamma, AnnForm form)
{
    if (!form.by_copies()) return;
    __shared__ AnnHalfLds L;
    const int lane = threadIdx.x, half = lane >> 5, r = lane & 31, sub = lane & 7, grp = lane >> 3;
    const int n_items = *n_blocks, pitch = 16 * kSteps;
    const float s = *scale, keep = 1.0f - kappa;
    const int stride = (int)gridDim.x, first = (int)blockIdx.x;
    if (first >= n_items) return;
    int waiting = 0;
    // what the next item begins with is read while this one is worked on: its queries and first members, and the descriptor after it
    auto query_of = [&](const int4& d) { return qlist[d.z + (r < d.w ? r : 0)]; };           // slots beyond nq repeat the first query
    auto member_of = [&](const int4& d, int c0) { return perm[d.x + c0 + (c0 + lane < d.y ? lane : 0)]; };
    int4 desc = blk_desc[first], ahead = blk_desc[min(first + stride, n_items - 1)];
    int next_q = query_of(desc), next_c = member_of(desc, 0);
    for (int item = first;; item += stride) {
        const bool last = item >= n_items;                 // (a round without an item: the pairs that still wait)
        const int S = last ? 1 : desc.y, nq = desc.w, my_q = next_q;
        const int4 now = desc;
        float tau = q_dist[(size_t)my_q * (size_t)K + (size_t)(K - 1)];
        int my_c = next_c;
        desc = ahead;
        ahead = blk_desc[min(item + 2 * stride, n_items - 1)];
        next_q = query_of(desc);
        next_c = member_of(desc, 0);
        int n_listed = 0;
        for (int c0 = 0; c0 < S; c0 += kMembers) {
            uint32_t left = 0;
            if (!last) {
                const int nc = min(kMembers, S - c0);
                const bool two = nc > 32;
                if (c0 > 0) {
                    my_c = member_of(now, c0);
                    tau = q_dist[(size_t)my_q * (size_t)K + (size_t)(K - 1)];
                }
                L.cid[lane] = my_c;
                if (half == 0) L.qid[r] = my_q;
                wave_lds_sync();
                // ---- 1.
                f32x16 g0, g1;
#pragma unroll
                for (int i = 0; i < 16; ++i) { g0[i] = 0.0f; g1[i] = 0.0f; }
                float nrm_q = 0.0f, nrm_0 = 0.0f, nrm_1 = 0.0f;
#pragma unroll
                for (int u0 = 0; u0 < kSteps; u0 += 4) {
                    wave_lds_drain();                      // (nothing of the tile is being read any more)
                    const int piece = sub ^ grp;           // of row 8 i + grp, for place sub
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int row = 8 * i + grp;
                        if (row < nc) load_to_lds(pc.rows + (size_t)L.cid[row] * (size_t)pitch + 16 * u0 + 8 * piece, &L.tile[64 * i]);
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int row = 8 * i + grp;
                        if (row < nq) load_to_lds(qc.rows + (size_t)L.qid[row] * (size_t)pitch + 16 * u0 + 8 * piece, &L.tile[64 * (8 + i)]);
                    }
                    wave_vm_drain();
                    f16x8 a[4], b[4], c[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        a[u] = __builtin_bit_cast(f16x8, L.tile[tile_at(64 + r, 2 * u + half)]);
                        b[u] = __builtin_bit_cast(f16x8, L.tile[tile_at(r, 2 * u + half)]);
                        c[u] = __builtin_bit_cast(f16x8, L.tile[tile_at(32 + r, 2 * u + half)]);
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        nrm_q = half_norm(a[u], nrm_q);
                        nrm_0 = half_norm(b[u], nrm_0);
                        g0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[u], a[u], g0, 0, 0, 0);
                        if (two) {
                            nrm_1 = half_norm(c[u], nrm_1);
                            g1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(c[u], a[u], g1, 0, 0, 0);
                        }
                    }
                }
                // a lane holds the squares of half of the dimensions of its row
                nrm_q += __shfl_xor(nrm_q, 32, 64);
                nrm_0 += __shfl_xor(nrm_0, 32, 64);
                nrm_1 += __shfl_xor(nrm_1, 32, 64);
                // (rows beyond nc and nq: whatever the tile held)
                const bool fine_0 = nrm_0 <= 3.0e38f, fine_1 = nrm_1 <= 3.0e38f;
                const float most = wave_max(fmaxf(fine_0 && r < nc ? nrm_0 : 0.0f, fine_1 && 32 + r < nc ? nrm_1 : 0.0f));
                if (half == 0) {
                    L.nrm[r] = fine_0 ? nrm_0 * keep : -INFINITY;           // (a row that is not finite is never dropped)
                    L.nrm[32 + r] = fine_1 ? nrm_1 * keep : -INFINITY;
                }
                wave_lds_sync();
                // ---- 2. accumulator i of lane l: member 8 (i / 4) + i % 4 + 4 (l / 32) of the block, query l % 32
                const float reach = __builtin_fmaf(s, sqrtf(tau / one_minus_gamma + 1e-30f),
                                                   __builtin_fmaf(err_rel, sqrtf(nrm_q) + sqrtf(most), 2.0f * err_abs)) * kJoinUp;
                const float line = nrm_q <= 3.0e38f ? __builtin_fmaf(-nrm_q, keep, reach * reach * kJoinUp) : INFINITY;
                auto screen = [&](const f32x16& g, int n0) {
                    uint32_t m = 0;
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const int n = n0 + 8 * i4 + 4 * half;
                        const float4 nn4 = *reinterpret_cast<const float4*>(&L.nrm[n]);
                        const float nn[4] = {nn4.x, nn4.y, nn4.z, nn4.w};
#pragma unroll
                        for (int x = 0; x < 4; ++x)
                            if (n + x < nc && !(__builtin_fmaf(-2.0f, g[4 * i4 + x], nn[x]) > line)) m |= 1u << (4 * i4 + x);
                    }
                    return m;
                };
                left = screen(g0, 0) | (two ? screen(g1, 32) << 16 : 0u);
                if (r >= nq) left = 0;
            }
            // the pairs of query r: those of lane r, then those of lane r + 32 (the list takes the place of the queries in the tile, which
            // evaluate() leaves alone)
            uint16_t* list = reinterpret_cast<uint16_t*>(&L.tile[kMembers * 8]);
            const int mine = __popc(left), other = __shfl_xor(mine, 32, 64);
            const int before = wave_excl_scan_i(half == 0 ? mine + other : 0), total = read_lane_i(before, 32);
            int at = __shfl(before, r, 64) + (half == 0 ? 0 : other);
            while (left) {
                const int i = __ffs(left) - 1;
                left &= left - 1;
                list[at++] = (uint16_t)(r | (2 * (i & ~15) + 8 * ((i & 15) >> 2) + (i & 3) + 4 * half) << 5);
            }
            n_listed += total;
            if (half == 0) L.tau[r] = tau;
            wave_lds_sync();
            for (int off = 0; off < total || (last && waiting > 0); off += kFlush) {
                const int take = max(0, min(kFlush, total - off));
                if (lane < take) {
                    const int e = list[off + lane], m = e & 31;
                    L.pend_q[waiting + lane] = L.qid[m];
                    L.pend_c[waiting + lane] = L.cid[e >> 5];
                    L.pend_tau[waiting + lane] = L.tau[m];
                }
                waiting += take;
                wave_lds_sync();
                if (waiting >= kFlush || last) {
                    evaluate(L, min(waiting, kFlush), points, queries, D, K, vec, q_idx, q_dist);
                    waiting = max(0, waiting - kFlush);
                    wave_lds_sync();
                    if (lane < waiting) {
                        L.pend_q[lane] = L.pend_q[kFlush + lane];
                        L.pend_c[lane] = L.pend_c[kFlush + lane];
                        L.pend_tau[lane] = L.pend_tau[kFlush + lane];
                    }
                    wave_lds_sync();
                }
            }
            wave_lds_sync();                               // done with cid and nrm
        }
        if (last) break;
        if (form.counts(item) && lane == 0)
            atomicAdd(form.word(item), ((unsigned long long)((unsigned)nq * (unsigned)S) << 32) | (unsigned)n_listed);
    }
}

}  // namespace

// The share of pairs (as ann_screen_share_q16) below which the bounds are made from the copies, 0: never.  The rows of the copies come in whole lines,
// but a pair that is left is one of 64 that wait together and costs more than in ann_screen.hip: trees late in a call, and rows that do not
// stay in the last cache (256 MB).  Per tree, fp32 rows -> copies, with the share that was left: 1M / 1M x 100 1797 -> 1895 us at 14 %, 1675 -> 1649 at
// 10 %, 1397 -> 1199 at 3.8 %; 500,000 / 500,000 x 128 785 -> 812 at 7.8 %, 724 -> 712 at 5.0 %, 671 -> 635 at 3 %; 300,000 / 500,000 x 100 702 -> 781 at 10 %,
// 617 -> 617 at 5.0 %, 550 -> 514 at 2.5 %; 200,000 / 300,000 x 100 405 -> 495, 330 -> 356, 311 -> 324; 60,000 / 250,000 x 128 276 -> 309, 230 -> 247, 216 -> 227.
// Tree t leaves about 72 / t per cent, and the copies take as long as two or three trees gain (300,000 / 500,000: seven): calls of fewer trees make none.
unsigned int ann_half_share_q16(int N, int NQ, int D, int n_trees, unsigned int share_q16)
{
    if (D <= 96 || D > 128 || share_q16 == 0) return 0;
    if (share_q16 == kScreenAlways) return n_trees > 1 ? kScreenAlways : 0;
    const size_t bytes = ((size_t)N + (size_t)NQ) * (size_t)D * sizeof(float);
    const bool beyond = bytes >= (size_t)640 << 20;
    if (bytes < (size_t)256 << 20 || n_trees < (beyond ? 12 : 30)) return 0;
    return std::min(share_q16, (unsigned int)((beyond ? 0.12 : 0.055) * 65536.0));
}

int launch_ann_screen_half(const JoinCopy& qc, const JoinCopy& pc, const float* points, const float* queries, int D, int K, const int* perm,
                           const int4* blk_desc, const int* n_blocks, int most_blocks, const int* qlist, int* q_idx, float* q_dist,
                           const AnnForm& form, hipStream_t stream)
{
    RSFK_CHECK(K >= 1 && K <= 64, "query-set search: screened form takes K up to 64");
    RSFK_CHECK(join_pitch(D) == 16 * kSteps, "query-set search: dimensions of the screened form by copies");
    const float kappa = (float)(16 * kSteps + 24) * (1.0f / 2097152.0f);            // (Dp + 24) 2^-21
    const float one_minus_gamma = 1.0f - (float)(D + 8) * (1.0f / 4194304.0f);
    RSFK_CHECK(one_minus_gamma > 0.5f, "query-set search: D too large for the screened form");
    int most = 16384;
    if (const char* e = std::getenv("RSFK_ANN_SCREEN_GROUPS")) most = std::max(1, std::atoi(e));       // for tests
    const unsigned grid = (unsigned)std::min(most, most_blocks);
    const bool vec = (D & 3) == 0 && ((reinterpret_cast<uintptr_t>(points) | reinterpret_cast<uintptr_t>(queries)) & 15) == 0;
    hipLaunchKernelGGL(k_ann_screen_half, dim3(grid), dim3(64), 0, stream, qc, pc, points, queries, D, K, vec, perm, blk_desc, n_blocks, qlist,
                       q_idx, q_dist, pc.scale(), kappa, join_err_rel(), join_err_abs(D), one_minus_gamma, form);
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
