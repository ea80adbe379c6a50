// One 64 x 64 tile of a bucket's pair matrix by a workgroup of 256 threads: the rows of its points on their way through
// LDS and the sequential fp32 chains.  Shared by the general bucket kernels (bucket_knn.hip) and the kernel that takes
// the buckets of several trees at once (bucket_knn_forest.hip).
#pragma once
#include "rsfk_common.hpp"

namespace rsfk {

constexpr int kTile = 64;          // points per tile side
constexpr int kDC = 32;            // dimensions staged per step
constexpr int kDCP = kDC + 4;      // LDS row pitch in floats: 9 x 16 B, odd => conflict-free b128 reads
constexpr int kDistPitch = kTile + 1;

// A thread's share (8 values of one row) of the rows ids[0..rows) x dims [d0, d0+32) on its way from memory to LDS:
// requested into registers first, so that the next 32 dimensions travel while these are being used.
struct StagedRows {
    float v[8];

    __device__ __forceinline__ void request(const int* __restrict__ ids, int rows, const float* __restrict__ points, int D,
                                            int d0, bool vec_ok)
    {
        const int t = threadIdx.x;
        const int r = t >> 2;            // 0..63
        const int seg = (t & 3) * 8;     // 0,8,16,24
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = 0.0f;
        if (r < rows && d0 + seg < D) {
            const float* src = points + (size_t)ids[r] * (size_t)D + d0 + seg;
            const int left = D - d0 - seg;
            if (left >= 8) {
                const float4 q0 = load_dims(src, 4, vec_ok);
                const float4 q1 = load_dims(src + 4, 4, vec_ok);
                v[0] = q0.x; v[1] = q0.y; v[2] = q0.z; v[3] = q0.w;
                v[4] = q1.x; v[5] = q1.y; v[6] = q1.z; v[7] = q1.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) if (e < left) v[e] = src[e];
            }
        }
    }

    // (zero filled outside the rows and beyond D)
    __device__ __forceinline__ void commit(float* __restrict__ dst) const
    {
        const int t = threadIdx.x;
        float4* d4 = reinterpret_cast<float4*>(dst + (t >> 2) * kDCP + (t & 3) * 8);
        d4[0] = make_float4(v[0], v[1], v[2], v[3]);
        d4[1] = make_float4(v[4], v[5], v[6], v[7]);
    }
};

// The chains of one tile: NRB x NCB blocks of 16 x 16 pairs (a thread has one pair of each block), DIAG: a tile on the
// diagonal, only the blocks on and above the diagonal.  Rows of the two tiles come through LDS 32 dimensions at a time,
// the next 32 on their way while these are used.
template <int NRB, int NCB, bool DIAG, typename Lds>
__device__ __forceinline__ void pair_tile_chains(Lds& L, const float* __restrict__ points, int D, int rows, int cols,
                                                 bool vec_ok, float (&acc)[4][4])
{
    const int tid = threadIdx.x;
    const int ty = tid >> 4, tx = tid & 15;
    StagedRows sa, sb;
    sa.request(L.ida, rows, points, D, 0, vec_ok);
    if (!DIAG) sb.request(L.idb, cols, points, D, 0, vec_ok);
    const float* B = DIAG ? L.a : L.b;
    for (int d0 = 0; d0 < D; d0 += kDC) {
        sa.commit(L.a);
        if (!DIAG) sb.commit(L.b);
        __syncthreads();
        if (d0 + kDC < D) {
            sa.request(L.ida, rows, points, D, d0 + kDC, vec_ok);
            if (!DIAG) sb.request(L.idb, cols, points, D, d0 + kDC, vec_ok);
        }
        const int nd = min(kDC, (D - d0 + 3) & ~3);          // (zeros beyond D)
#pragma unroll 2
        for (int dd = 0; dd < nd; dd += 4) {
            float4 av[NRB], bv[NCB];
#pragma unroll
            for (int r = 0; r < NRB; ++r) av[r] = *reinterpret_cast<const float4*>(&L.a[(ty + 16 * r) * kDCP + dd]);
#pragma unroll
            for (int c = 0; c < NCB; ++c) bv[c] = *reinterpret_cast<const float4*>(&B[(tx + 16 * c) * kDCP + dd]);
#pragma unroll
            for (int r = 0; r < NRB; ++r) {
#pragma unroll
                for (int c = 0; c < NCB; ++c) {
                    if (DIAG && c < r) continue;
                    float df;
                    df = av[r].x - bv[c].x; acc[r][c] = __builtin_fmaf(df, df, acc[r][c]);
                    df = av[r].y - bv[c].y; acc[r][c] = __builtin_fmaf(df, df, acc[r][c]);
                    df = av[r].z - bv[c].z; acc[r][c] = __builtin_fmaf(df, df, acc[r][c]);
                    df = av[r].w - bv[c].w; acc[r][c] = __builtin_fmaf(df, df, acc[r][c]);
                }
            }
        }
        __syncthreads();
    }
}

// ... with the number of 16 x 16 blocks the tile really has (off the diagonal tile I is full: J > I; on it rows == cols)
template <typename Lds>
__device__ __forceinline__ void pair_tile(Lds& L, const float* __restrict__ points, int D, int rows, int cols, bool diag,
                                          bool vec_ok, float (&acc)[4][4])
{
    const int nrb = (rows + 15) >> 4, ncb = (cols + 15) >> 4;
    if (diag) {
        switch (nrb) {
        case 1: pair_tile_chains<1, 1, true>(L, points, D, rows, cols, vec_ok, acc); break;
        case 2: pair_tile_chains<2, 2, true>(L, points, D, rows, cols, vec_ok, acc); break;
        case 3: pair_tile_chains<3, 3, true>(L, points, D, rows, cols, vec_ok, acc); break;
        default: pair_tile_chains<4, 4, true>(L, points, D, rows, cols, vec_ok, acc); break;
        }
    } else {
        switch (ncb) {
        case 1: pair_tile_chains<4, 1, false>(L, points, D, rows, cols, vec_ok, acc); break;
        case 2: pair_tile_chains<4, 2, false>(L, points, D, rows, cols, vec_ok, acc); break;
        case 3: pair_tile_chains<4, 3, false>(L, points, D, rows, cols, vec_ok, acc); break;
        default: pair_tile_chains<4, 4, false>(L, points, D, rows, cols, vec_ok, acc); break;
        }
    }
}

}  // namespace rsfk
