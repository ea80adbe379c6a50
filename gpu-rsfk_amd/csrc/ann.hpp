// Query-set search, one tree after the other: what the two forms of the bucket step share (ann.hip, ann_screen.hip).
#pragma once
#include "rsfk_common.hpp"
#include "join_copy.hpp"
#include "wave64.hpp"
#include <cmath>

namespace rsfk {

constexpr int kAnnDirect = 16;        // queries of a work item: a workgroup that evaluates every pair
constexpr int kAnnScreen = 32;        // ... a wavefront that bounds the pairs on the matrix cores first
constexpr int kAnnStatWords = 8;      // of a tree: pairs << 32 | pairs that had to be evaluated, of a sample of the work items

// The form a tree's buckets are searched in, as the tree before it left its numbers behind (prev; null: the direct form,
// which also puts rows in order that the caller passed in unsorted).
struct AnnForm {
    const unsigned long long* prev;
    unsigned long long* stats;        // this tree's own (null: none are kept)
    unsigned int share_q16;           // a screened form when fewer than share_q16 / 65536 of the pairs had to be evaluated,
    unsigned int half_q16;            // the one by float16 copies when fewer than this (at most share_q16; 0: never)
    int shift;                        // one work item in 2^shift is counted

    __device__ __forceinline__ bool screened() const { return below(share_q16); }
    __device__ __forceinline__ bool by_copies() const { return half_q16 != 0 && below(half_q16); }
    __device__ __forceinline__ bool below(unsigned int share) const
    {
        if (prev == nullptr) return false;
        if (share == kScreenAlways) return true;
        unsigned long long pairs = 0, listed = 0;
#pragma unroll
        for (int i = 0; i < kAnnStatWords; ++i) {
            pairs += prev[i] >> 32;
            listed += prev[i] & 0xffffffffull;
        }
        return (listed << 16) < pairs * share;
    }
    __device__ __forceinline__ bool counts(int item) const { return stats != nullptr && (item & ((1 << shift) - 1)) == 0; }
    __device__ __forceinline__ unsigned long long* word(int item) const { return &stats[(item >> shift) & (kAnnStatWords - 1)]; }
};

// Side tests by rounded hyperplanes (ann_top.hip, k_route_low of ann.hip).  x~ = float16(s (x - mu)), the rows of a JoinCopy of the queries;
// n~ = float16(K n / |n|), K = 2^8, what is below 2^-14 set to zero; b~ = (offset - n.mu) K s / |n| in 64 bits, rounded.  For t = n~.x~ - b~
//   |t - K s (n.x - offset) / |n| | <=  |n~ - K n / |n|| |x~|  +  K |s (x - mu) - x~|  +  kappa (K |x~| + |b~|)  +  2^-22 |b~|
// (Cauchy-Schwarz; kappa for the accumulation), and the exact test sums n.x in fp32 to within gamma |n| |x|.  With 2^-11 (and what is
// set to zero) for the first term and the measured error of the row for the second, all but the terms of b~ depend on the query alone
// (query()), and a side is certain when |t| is above the sum.  Hyperplanes and queries for which a sum of the exact test could leave
// the range of fp32, or be lost below it, are never certain.
struct SideBound {
    static constexpr float kUnit = 256.0f;                    // K
    float rel = 0, err = 0, gamma = 0, kappa = 0;

    SideBound() = default;
    explicit SideBound(int D)
    {
        kappa = (float)(((D + 15) & ~15) + 16) / 2097152.0f;
        gamma = (float)(D + 64) / 8388608.0f;
        err = kUnit * (1.0f + 1.0f / 512.0f);
        rel = kUnit * (1.003f / 2048.0f) + std::sqrt((float)D) / 16384.0f;     // (the second term: what is set to zero)
    }
    __device__ __forceinline__ float of_offset() const { return kappa + 1.0f / 4194304.0f; }        // times |b~|
    // s: scale of the copy, mu_len >= |mu|; infinite: no side of this query is certain
    __device__ __forceinline__ float query(float norm, float row_err, float s, float mu_len) const
    {
        const float X = sqrtf(norm) * (1.0f + 1.0f / 1024.0f), far = X + row_err + mu_len * s;
        // (the last terms: what a query is off by at least, and products that underflow; |n| is above 1e-12)
        const float z = rel * X + err * (row_err + gamma * far) + kappa * kUnit * X + 1e-6f + kUnit * s * 1e-30f;
        return z < 1e30f && far < 1e15f * s ? z : INFINITY;
    }
};

// Of a hyperplane, by one wavefront: lanes' own dimensions d = lane, lane + 64, ... of the rounded normal are unit * n_d.
struct RoundedPlane { float unit, b; bool sound; };
__device__ __forceinline__ RoundedPlane rounded_plane(const float* __restrict__ x1, const float* __restrict__ x2, int D, float offset,
                                                      const float* __restrict__ mu, float s)
{
    double len2 = 0.0, n_mu = 0.0;
    for (int d = lane_id(); d < D; d += 64) {
        const double nd = (double)(x1[d] - x2[d]);
        len2 += nd * nd;
        n_mu += nd * (double)mu[d];
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        len2 += __shfl_xor(len2, o, 64);
        n_mu += __shfl_xor(n_mu, o, 64);
    }
    const double per = (double)SideBound::kUnit / sqrt(len2);
    RoundedPlane p;
    p.unit = (float)per;
    p.b = (float)(((double)offset - n_mu) * per * (double)s);
    p.sound = len2 > 1e-24 && len2 < 1e30 && fabsf(offset) < 1e30f && fabsf(p.b) < 1e30f;      // (false for NaN)
    return p;
}
__device__ __forceinline__ uint16_t rounded_value(float nd, const RoundedPlane& p)
{
    const float v = p.sound ? nd * p.unit : 0.0f;
    const _Float16 h = fabsf(v) < 6.103515625e-5f ? (_Float16)0.0f : (_Float16)v;
    return __builtin_bit_cast(uint16_t, h);
}

// ann_screen.hip.  blk_desc: {start and size of the bucket in perm, first query in qlist, queries}, *n_blocks of them, at most
// most_blocks.  Works only when form.screened().  K at most 64, rows sorted.
int launch_ann_screen(const float* points, const float* queries, int D, int K, const int* perm, const int4* blk_desc,
                      const int* n_blocks, int most_blocks, const int* qlist, int* q_idx, float* q_dist, const AnnForm& form,
                      hipStream_t stream);
// ann_screen_half.hip: the same by copies of the queries and of the points with the same mu and s; only when form.by_copies(), when the one above leaves
int launch_ann_screen_half(const JoinCopy& qc, const JoinCopy& pc, const float* points, const float* queries, int D, int K, const int* perm,
                           const int4* blk_desc, const int* n_blocks, int most_blocks, const int* qlist, int* q_idx, float* q_dist,
                           const AnnForm& form, hipStream_t stream);

}  // namespace rsfk
