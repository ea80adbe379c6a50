// What the join (explore_join.hip) leaves of the distance of a pair it marked, and what the merge kernels (explore.hip) read from it.
//
// All lengths are in the units of the float16 copy (join_copy.hpp: s times those of the points).  For a pair (p, c) the join has
// least = d~ - E1 <= d~(real) and t = max(0, sqrt(least) - e_p - e_c), a lower bound of the distance of the points.  Kept is
//   code = 1 + min(65534, floor(65534 t / span_p)),   0: nothing is known (a row that is not finite),
// span_p = the bar of point p (k_join_bars), or four times the largest distance from the centre where its row is not full.  A code stands
// for an interval: the pair's exact distance (the fp32 chain) is at least what its lower end gives, and at most what its upper end
// gives with the errors put on instead of taken off:
//   sqrt(d~(real)) <= sqrt((t + e_p + e_c)^2 + 2 E1),   sqrt(d) <= that + e_p + e_c,   chain <= d (1 + gamma),
// with the largest e_c and E1 of any point, or of one no farther than 2 span.  So the codes of a point's candidates tell, before any exact
// distance is known, how far its row will reach at most: K of its entries and candidates lie below.  (Codes of 65535 have no upper
// end.)
#pragma once
#include "rsfk_common.hpp"

namespace rsfk {

constexpr float kJoinUp = 1.0f + 1.0f / 1048576.0f, kJoinDown = 1.0f - 1.0f / 1048576.0f;
constexpr int kCodeTop = 65535;

struct JoinBounds {
    const uint16_t* codes = nullptr;   // N*K*KP words by graph entry and neighbour slot, or null
    const float* bars = nullptr;       // bar of a point (k_join_bars)
    const float* norms = nullptr;      // JoinCopy::norms
    const float* scale = nullptr;      // JoinCopy::scale: s, largest norm, largest error
    float kappa = 0.0f;                // E1 = kappa S
    float one_minus_gamma = 1.0f;
    float any_rel = 0.0f, any_abs = 0.0f;   // e <= any_rel |row| + any_abs of any row
};

__device__ __forceinline__ float join_span(float bar, float most_norm)
{
    return bar <= 3.0e38f ? bar : 4.0f * sqrtf(most_norm);
}

// What the rounding of any row took at most, from the norm of the row and from the largest that was measured (most_err).
__device__ __forceinline__ float join_err(float norm, float any_rel, float any_abs, float most_err)
{
    return fminf(__builtin_fmaf(any_rel, __builtin_amdgcn_sqrtf(norm), any_abs), most_err);
}

// per = 65534 / span
__device__ __forceinline__ uint32_t join_code(float least, float e_p, float e_c, float per)
{
    if (!(least <= 3.0e38f)) return 0u;
    // (2^-20: one unit of the square root and the roundings here)
    const float t = __builtin_fmaf(__builtin_amdgcn_sqrtf(fmaxf(least, 0.0f)), kJoinDown, -(e_p + e_c) * kJoinUp);
    return 1u + min(65534u, (uint32_t)(fmaxf(t, 0.0f) * (per * kJoinDown)));
}

// The codes of one point, as seen from its row.
struct CodeReader {
    float per, len, inv_s, s, omg, E, E1;

    __device__ __forceinline__ CodeReader(const JoinBounds& b, int p)
    {
        const float norm = b.norms[p], span = join_span(b.bars[p], b.scale[1]), root = sqrtf(norm);
        s = *b.scale;
        inv_s = 1.0f / s;
        omg = b.one_minus_gamma;
        per = 65534.0f / span;
        len = span / 65534.0f;
        const float far = fminf(root + 2.0f * span, sqrtf(b.scale[1]) * kJoinUp);        // lengths of other points
        E = (join_err(norm, b.any_rel, b.any_abs, b.scale[2]) + fminf(b.any_rel * far + b.any_abs, b.scale[2])) * (1.0f + 1.0f / 131072.0f);
        E1 = 2.0f * kJoinUp * b.kappa * (norm + far * far);
        if (!((span + E) * (span + E) + E1 < 3.9f * span * span)) E = INFINITY;       // (what it leads to does not stay within 2 span)
    }
    // a pair with a code above this has an exact distance above tau
    __device__ __forceinline__ int last_code(float tau) const
    {
        const float x = s * sqrtf((tau + 1e-30f) / omg) * (per * (1.0f + 1.0f / 131072.0f));
        return x < 65532.0f ? (int)x + 2 : kCodeTop;
    }
    // the exact distance of a pair with this code (1..65534) is at most
    __device__ __forceinline__ float reach(int code) const
    {
        const float a = __builtin_fmaf((float)code, len * (1.0f + 1.0f / 262144.0f), E);
        const float b = (sqrtf(__builtin_fmaf(a, a, E1)) + E) * inv_s;
        return b * b * ((2.0f - omg) * (1.0f + 1.0f / 131072.0f)) + 1e-30f;
    }
    // a code whose reach is at least dist (a few more than the first one), or above all codes
    __device__ __forceinline__ int code_of(float dist) const
    {
        if (!(dist <= 3.4e38f)) return 0x7ffffffe;
        const float y = s * sqrtf(dist) - E, a = sqrtf(fmaxf(__builtin_fmaf(y, y, -E1), 0.0f));
        const float x = ((y > 0.0f ? a : 0.0f) - E) * per;
        return x < 65500.0f ? max((int)x, 0) + 4 : 0x7ffffffe;
    }
};

}  // namespace rsfk
