// bfloat16 screening copy of the points.
//
// Row p of the copy holds the coordinates of point p rounded to bfloat16 (round to
// nearest even), padded with zeros to a multiple of 8 values so that rows and
// 16-byte pieces of rows are aligned; norms[p] = sum of the squares of the rounded
// coordinates.  The copy halves the bytes of every pass that only has to decide an
// inequality (side of a hyperplane, "is this candidate closer than the row
// maximum"): the kernels evaluate the inequality on the copy with a rigorous error
// bound and fall back to the fp32 row inside the band where the bound cannot
// decide, so results are those of the fp32 arithmetic.
#pragma once
#include "rsfk_common.hpp"

namespace rsfk {

// Row pitch in values: rows start on 64-byte boundaries so that a row touches the
// minimum number of memory sectors.  bf16_valid(D) <= bf16_pitch(D) is the length the
// kernels loop over (whole 16-byte pieces); values between D and the pitch are zero.
__host__ __device__ inline int bf16_pitch(int D) { return (D + 31) & ~31; }
__host__ __device__ inline int bf16_valid(int D) { return (D + 7) & ~7; }

struct Bf16Copy {
    uint16_t* rows = nullptr;     // N x bf16_pitch(D)
    float* norms = nullptr;       // N
};

// 8-bit screening copy of the points, used by the side test of the tree build when the rows have a narrow
// range of values (half the bytes of the bfloat16 copy).
//
// Row p, q8_pitch(D) bytes on a 64-byte boundary: a 16-byte header (pad, lo, scale, e1 as four floats), then one
// byte per coordinate, q_d = round((x_d - lo) / scale) in 0..255 with lo = min_d x_d and scale = (max_d x_d - lo) / 255,
// zeros up to the end of the row.  e1 bounds what the quantisation can do to a dot product per unit of a
// length L(n) of the other vector: for any n, |n.x - (lo sum_d n_d + scale sum_d n_d q_d)| <= e1 L(n), including
// the fp32 evaluation of either side with at most D/8-term chains (see k_to_q8).  L(n) = min(||n||_1, kRmsShare sqrt(D) ||n||_2):
// the first factor goes with the largest error of a coordinate, the second (Cauchy and Schwarz) with the root of their mean square,
// which is 1 / sqrt(3) of the largest where coordinates fall anywhere between two steps; e1 is the larger of the largest error and
// 1 / kRmsShare of that root, so either holds.  For normals whose components spread like those of a uniform or a normal distribution
// L(n) is 0.71..0.73 ||n||_1 (points left to the exact test: 1M x 100 uniform 3.77 -> 2.74 %, 1M x 256 in clusters 12.3 -> 9.1 %; trees of the former 24.4 -> 23.5 ms for 50, of the latter 29.4 -> 26.4 for 20).  mean_rho (host, after
// q8_copy_fill has completed) compares the bound by the largest error, per unit of ||n||_1, with the corresponding quantity of the bfloat16 copy,
// 2^-8 mean_d |x_d|, averaged over the rows: the 8-bit copy pays off while it is below about 6.  (Not e1, which can be 1.72 times that where
// L(n) makes up for it.  One tree of 5,000 x 4096 normal points, 5.9 by the one and 6.0 by the other: 13.3 ms by the 8-bit copy, 14.9 by the bfloat16 copy.  Since
// L(n) the times of the two meet at 6 to 7 for 784 dimensions, 10 for 256, beyond 12 for 100 and fewer.)
__host__ __device__ inline int q8_pitch(int D) { return (16 + D + 63) & ~63; }
__host__ __device__ inline int q8_padded(int D) { return (D + 15) & ~15; }      // coordinates in whole 16-byte pieces

constexpr int kQ8MostGrid = 8192;       // workgroups (and parts of the statistic) of the kernel that makes the copy
struct Q8Copy {
    uint8_t* rows = nullptr;      // N x q8_pitch(D)
    float* rho_parts = nullptr;   // device, n_parts of them: sums over rows of e1 / (2^-8 mean |x_d|)
    int n_parts = 0;
};

// The screens of the side tests decide where margin > band: margin = |approximate n.x - offset|, band = what the approximation and
// the exact fp32 evaluation can differ by.  Where a sum of the exact evaluation could leave the range of fp32 (its comparison
// then has a side of its own) they must not decide, and what underflow does has to be in the band.
// 8-bit copy: not used at all when a finite row has a coordinate beyond q8_most(D) (mean_rho is infinite then).  Up to there
// |n.x| <= 2 D q8_most^2 = 1e38, and neither evaluation nor the offset can overflow; a row or a normal that is not finite has a
// band that is NaN or infinite.  e1 has kQ8Least in it and L(n) kNormalLeast, whose product is above the
// 2e-45 D that underflow amounts to.
// bfloat16 copy: sum |n_d||x_d|, which is part of the band, is compared with 1e38 at every point.  (The same for the 8-bit copy, or
// limits per row and per hyperplane: tail kernel and chains of 20,000 x 64, 50 trees 1.02 -> 1.06 and 1.04 ms.)
constexpr float kQ8Least = 1e-21f, kNormalLeast = 1e-18f;
constexpr float kRmsShare = 0.58f;
inline float q8_most(int D) { return 7.07e18f / __builtin_sqrtf((float)D); }

int q8_copy_alloc(Q8Copy* c, int N, int D);
void q8_copy_free(Q8Copy* c);
int q8_copy_fill(Q8Copy& c, const float* points, int N, int D, hipStream_t stream);
int q8_copy_mean_rho(const Q8Copy& c, int N, float* mean_rho, hipStream_t stream);     // synchronises the stream

size_t bf16_copy_bytes(int N, int D);
int bf16_copy_alloc(Bf16Copy* c, int N, int D);
void bf16_copy_free(Bf16Copy* c);
int bf16_copy_fill(const Bf16Copy& c, const float* points, int N, int D, hipStream_t stream);

}  // namespace rsfk
