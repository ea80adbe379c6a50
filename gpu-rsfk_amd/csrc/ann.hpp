// Query-set search, one tree after the other: what the two forms of the bucket step share (ann.hip, ann_screen.hip).
#pragma once
#include "rsfk_common.hpp"

namespace rsfk {

constexpr int kAnnDirect = 16;        // queries of a work item: a workgroup that evaluates every pair
constexpr int kAnnScreen = 32;        // ... a wavefront that bounds the pairs on the matrix cores first
constexpr int kAnnStatWords = 8;      // of a tree: pairs << 32 | pairs that had to be evaluated, of a sample of the work items

// The form a tree's buckets are searched in, as the tree before it left its numbers behind (prev; null: the direct form,
// which also puts rows in order that the caller passed in unsorted).
struct AnnForm {
    const unsigned long long* prev;
    unsigned long long* stats;        // this tree's own (null: none are kept)
    unsigned int share_q16;           // the screened form when fewer than share_q16 / 65536 of the pairs had to be evaluated
    int shift;                        // one work item in 2^shift is counted

    __device__ __forceinline__ bool screened() const
    {
        if (prev == nullptr) return false;
        if (share_q16 == kScreenAlways) return true;
        unsigned long long pairs = 0, listed = 0;
#pragma unroll
        for (int i = 0; i < kAnnStatWords; ++i) {
            pairs += prev[i] >> 32;
            listed += prev[i] & 0xffffffffull;
        }
        return (listed << 16) < pairs * share_q16;
    }
    __device__ __forceinline__ bool counts(int item) const { return stats != nullptr && (item & ((1 << shift) - 1)) == 0; }
    __device__ __forceinline__ unsigned long long* word(int item) const { return &stats[(item >> shift) & (kAnnStatWords - 1)]; }
};

// ann_screen.hip.  blk_desc: {start and size of the bucket in perm, first query in qlist, queries}, *n_blocks of them, at most
// most_blocks.  Works only when form.screened().  K at most 64, rows sorted.
int launch_ann_screen(const float* points, const float* queries, int D, int K, const int* perm, const int4* blk_desc,
                      const int* n_blocks, int most_blocks, const int* qlist, int* q_idx, float* q_dist, const AnnForm& form,
                      hipStream_t stream);

}  // namespace rsfk
