// 16-bit copy of the points for the join of the exploration (explore_join.hip), and of queries and points for the query-set search: the
// way of the queries through the trees (ann_top.hip, k_route_low of ann.hip) and the bounds in their buckets (ann_screen.hip).
//
// Row p holds s (x - mu) in float16 (round to nearest; below 2^-14, the least normal number, zero), mu the column means and s a
// power of two, padded with zeros to join_pitch(D) values; norms[p] = sum of the squares of the values as rounded, errs[p] >=
// |s (x_p - mu) - row p| as vectors, measured when the row is made.  Distances do not change under a common shift, and what rounding
// takes shrinks with the norms.  s is such that the largest value lies between 2^12 and 2^15: nothing overflows, and values down to
// 2^-26 of the largest keep their 11 bits.  (bfloat16 needs no s, but keeps 8 bits: at the same bytes its rounding is eight times as
// large.)  A row that is not finite has a norm that is not finite.
#pragma once
#include "rsfk_common.hpp"
#include <cmath>

namespace rsfk {

// rows start on 64-byte boundaries; the kernels take 16 dimensions per step
__host__ __device__ inline int join_pitch(int D) { return (D + 31) & ~31; }

constexpr int kJoinMostGrid = 8192;     // workgroups (and parts) of the kernel that makes the copy

struct JoinCopy {
    uint16_t* rows = nullptr;     // N x join_pitch(D)
    float* norms = nullptr;       // N, in units of s^2
    float* errs = nullptr;        // N, in units of s
    float* mu = nullptr;          // column means, then (s, largest norm, largest error of the finite rows, a bound of |mu|), then D words of working memory
    float2* parts = nullptr;      // n_parts: largest norm and error of the finite rows a workgroup made (k_join_bars completes them)
    int n_parts = 0;
    int D = 0;
    float* scale() const { return mu + D; }
    float* mu_len() const { return mu + D + 3; }
};

// optional: as blocks the caller can do without (ws_try_alloc)
int join_copy_alloc(JoinCopy* c, int N, int D, bool optional = false);
void join_copy_free(JoinCopy* c);
// like (null: none): the copy whose mu and s these rows take too; what overflows then is not finite
int join_copy_fill(JoinCopy& c, const float* points, int N, int D, hipStream_t stream, const JoinCopy* like = nullptr);

// Rounding of any row, errs <= rel |row| + abs: 2^-11 of a value, 2^-14 of one set to zero, and errs' own terms (3e-3 covers these and the
// root).
inline float join_err_rel() { return 1.003f / 2048.0f; }
inline float join_err_abs(int D) { return 1.001f * std::sqrt((float)D) / 16384.0f + 1e-6f; }

// acc + the squares of eight values of a row
__device__ __forceinline__ float half_norm(__attribute__((ext_vector_type(8))) _Float16 v, float acc)
{
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const f16x2 h = {v[i], v[i + 1]};
        acc = __builtin_amdgcn_fdot2(h, h, acc, false);
    }
    return acc;
}

}  // namespace rsfk
