#include "join_copy.hpp"
#include "wave64.hpp"
#include <algorithm>

namespace rsfk {

namespace {

// magnitude as ordered bits; what is not finite does not count
__device__ __forceinline__ uint32_t spread_bits(float x)
{
    const uint32_t b = __float_as_uint(x) & 0x7fffffffu;
    return b < 0x7f800000u ? b : 0u;
}
__device__ __forceinline__ float finite_or_zero(float x) { return fabsf(x) <= 3.0e38f ? x : 0.0f; }

__global__ void k_col_clear(uint32_t* __restrict__ a, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0u;
}

// Column sums of the rows less the first one (columns whose first value is not finite: as they are): a workgroup adds up its share
// of the rows, 256 columns at a time, and adds the result to sum[]; the largest magnitude goes to spread[].
__global__ __launch_bounds__(256) void k_col_sum(const float* __restrict__ points, int N, int D, float* __restrict__ sum,
                                                 uint32_t* __restrict__ spread)
{
    const int rows_per = (N + gridDim.x - 1) / gridDim.x;
    const int r0 = blockIdx.x * rows_per, r1 = min(N, r0 + rows_per);
    for (int d = threadIdx.x; d < D; d += 256) {
        const float ref = finite_or_zero(points[d]);
        float acc = 0.0f;
        uint32_t far = 0u;
        const float* src = points + d;
        int r = r0;
        for (; r + 7 < r1; r += 8) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = src[(size_t)(r + u) * (size_t)D];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float x = v[u] - ref;
                acc += x;
                far = max(far, spread_bits(x));
            }
        }
        for (; r < r1; ++r) {
            const float x = src[(size_t)r * (size_t)D] - ref;
            acc += x;
            far = max(far, spread_bits(x));
        }
        atomicAdd(&sum[d], acc);
        atomicMax(&spread[d], far);
    }
}

// The same for D <= 128: the workgroup reads m = 256 / D whole rows per step (thread t: row t / D of the step, column
// t % D, so its column never changes), eight steps in flight; the threads of a column are added up in LDS.
__global__ __launch_bounds__(256) void k_col_sum_narrow(const float* __restrict__ points, int N, int D, float* __restrict__ sum,
                                                        uint32_t* __restrict__ spread)
{
    __shared__ float part[256];
    __shared__ uint32_t part_far[256];
    const int m = 256 / D;
    const int rows_per = (N + gridDim.x - 1) / gridDim.x;
    const int r0 = blockIdx.x * rows_per, r1 = min(N, r0 + rows_per);
    const int sub = threadIdx.x / D, col = threadIdx.x - sub * D;
    const float ref = finite_or_zero(points[col]);
    float acc = 0.0f;
    uint32_t far = 0u;
    if (sub < m) {
        const float* src = points + col;
        int r = r0 + sub;
        for (; r + 7 * m < r1; r += 8 * m) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = src[(size_t)(r + u * m) * (size_t)D];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const float x = v[u] - ref;
                acc += x;
                far = max(far, spread_bits(x));
            }
        }
        for (; r < r1; r += m) {
            const float x = src[(size_t)r * (size_t)D] - ref;
            acc += x;
            far = max(far, spread_bits(x));
        }
    }
    part[threadIdx.x] = acc;
    part_far[threadIdx.x] = far;
    __syncthreads();
    if ((int)threadIdx.x < D) {
        float t = 0.0f;
        far = 0u;
        for (int u = 0; u < m; ++u) {
            t += part[u * D + threadIdx.x];
            far = max(far, part_far[u * D + threadIdx.x]);
        }
        atomicAdd(&sum[threadIdx.x], t);
        atomicMax(&spread[threadIdx.x], far);
    }
}

// One workgroup: sums -> means (where a sum is not finite, the first value: any shift is a valid one), and s = 2^(14 - e) with 2^e
// above the largest distance f from the first row: |x - mu| is at most 2 f and what the sums lose, so s |x - mu| < 2^15 (1 + small);
// exponents beyond what fp32 holds on either side are cut off.
__global__ __launch_bounds__(256) void k_col_mean(const float* __restrict__ points, float* __restrict__ mu,
                                                  const uint32_t* __restrict__ spread, float* __restrict__ scale, int D, float inv_n)
{
    __shared__ uint32_t part[256];
    __shared__ float part_q[256];
    uint32_t far = 0u;
    float q = 0.0f;
    for (int d = threadIdx.x; d < D; d += 256) {
        const float m = finite_or_zero(points[d]) + finite_or_zero(mu[d] * inv_n);
        mu[d] = m;
        q = __builtin_fmaf(m, m, q);
        far = max(far, spread[d]);
    }
    part[threadIdx.x] = far;
    part_q[threadIdx.x] = q;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            part[threadIdx.x] = max(part[threadIdx.x], part[threadIdx.x + o]);
            part_q[threadIdx.x] += part_q[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        scale[3] = sqrtf(part_q[0]) * (1.0f + 1.0f / 1024.0f) + 1e-18f;
        const int e = (int)(part[0] >> 23) - 126;                          // f < 2^e
        *scale = __uint_as_float((uint32_t)(127 + max(-100, min(100, 14 - e))) << 23);
    }
}

__global__ __launch_bounds__(256) void k_col_take(const float* __restrict__ from, float* __restrict__ to, int n)
{
    for (int i = threadIdx.x; i < n; i += 256) to[i] = from[i];
}

// LPR lanes per row (64 / LPR rows per wavefront), each four dimensions at a time.  Streaming; 10M x 32 (8 lanes per row) 2.0 GB in
// 0.35 ms, 5.7 TB/s (a wavefront per row, a value per lane: 1.13); 1M x 256 0.26 (0.42), 1M x 100 0.12 (0.22).
template <int LPR, bool WHOLE>
__global__ __launch_bounds__(256) void k_to_join(const float* __restrict__ points, uint16_t* __restrict__ out, float* __restrict__ norms,
                                                 float* __restrict__ errs, float2* __restrict__ parts, const float* __restrict__ mu,
                                                 const float* __restrict__ scale, int N, int D, int pitch)
{
    constexpr int kRowsPerWave = 64 / LPR;
    const int lane = threadIdx.x & 63, sub = lane / LPR, l = lane - sub * LPR;
    const int wave_global = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int n_waves = (gridDim.x * blockDim.x) >> 6;
    const float s = *scale;
    const float sums = 1.0f + (float)(D + 16) * (1.0f / 16777216.0f);      // sums of D squares, in any order
    float most_q = 0.0f, most_e = 0.0f;
    for (int rb = wave_global * kRowsPerWave; rb < N; rb += n_waves * kRowsPerWave) {
        const int r = rb + sub;
        const bool row_ok = r < N;
        const float* src = points + (size_t)(row_ok ? r : 0) * (size_t)D;
        uint16_t* dst = out + (size_t)(row_ok ? r : 0) * (size_t)pitch;
        float q = 0.0f, e = 0.0f;
        for (int d = 4 * l; d < pitch; d += 4 * LPR) {
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (d < D) {
                const float4 x = load_dims(src + d, D - d, WHOLE), m = load_dims(mu + d, D - d, false);
                v[0] = (x.x - m.x) * s;
                v[1] = (x.y - m.y) * s;
                v[2] = (x.z - m.z) * s;
                v[3] = (x.w - m.w) * s;
            }
            uint16_t h[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const _Float16 f = fabsf(v[c]) < 6.103515625e-5f ? (_Float16)0.0f : (_Float16)v[c];
                h[c] = __builtin_bit_cast(uint16_t, f);
                const float g = (float)f, w = v[c] - g;                    // exact: the low bits of v
                q = __builtin_fmaf(g, g, q);
                e = __builtin_fmaf(w, w, e);
            }
            if (row_ok) *reinterpret_cast<uint2*>(dst + d) = make_uint2(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16);
        }
#pragma unroll
        for (int o = 1; o < LPR; o <<= 1) {
            q += __shfl_xor(q, o, 64);
            e += __shfl_xor(e, o, 64);
        }
        // fl(x - mu) is within 2^-24 |fl(x - mu)| of x - mu, which is at most 1.1 |row| and what was set to zero (1e-8 stands for it)
        e = sums * (sqrtf(e) + (1.2f / 16777216.0f) * sqrtf(q)) + 1e-8f;
        if (row_ok && l == 0) {
            norms[r] = q;
            errs[r] = e;
        }
        if (row_ok && q <= 3.0e38f) {
            most_q = fmaxf(most_q, q);
            most_e = fmaxf(most_e, e);
        }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        most_q = fmaxf(most_q, __shfl_xor(most_q, o, 64));
        most_e = fmaxf(most_e, __shfl_xor(most_e, o, 64));
    }
    __shared__ float2 part[4];
    if (lane == 0) part[threadIdx.x >> 6] = make_float2(most_q, most_e);
    __syncthreads();
    if (threadIdx.x == 0)
        parts[blockIdx.x] = make_float2(fmaxf(fmaxf(part[0].x, part[1].x), fmaxf(part[2].x, part[3].x)),
                                        fmaxf(fmaxf(part[0].y, part[1].y), fmaxf(part[2].y, part[3].y)));
}

}  // namespace

int join_copy_alloc(JoinCopy* c, int N, int D, bool optional)
{
    c->D = D;
    const auto get = [optional](void* p, size_t bytes) {
        void** out = reinterpret_cast<void**>(p);
        return optional ? ws_try_alloc(out, bytes) : ws_alloc(out, bytes);
    };
    if (get(&c->mu, ((size_t)2 * D + 4) * sizeof(float))) return 1;
    if (get(&c->parts, kJoinMostGrid * sizeof(float2))) return 1;
    if (get(&c->rows, std::max<size_t>((size_t)N * join_pitch(D) * 2, 16))) return 1;
    if (get(&c->norms, std::max<size_t>((size_t)N * 4, 16))) return 1;
    if (get(&c->errs, std::max<size_t>((size_t)N * 4, 16))) return 1;
    return 0;
}

void join_copy_free(JoinCopy* c)
{
    ws_free(c->rows);
    ws_free(c->norms);
    ws_free(c->errs);
    ws_free(c->mu);
    ws_free(c->parts);
    *c = JoinCopy();
}

int join_copy_fill(JoinCopy& c, const float* points, int N, int D, hipStream_t stream, const JoinCopy* like)
{
    float* scale = c.mu + D;
    uint32_t* spread = reinterpret_cast<uint32_t*>(scale + 4);
    if (like) {
        hipLaunchKernelGGL(k_col_take, dim3(1), dim3(256), 0, stream, like->mu, c.mu, D + 4);
    } else {
        hipLaunchKernelGGL(k_col_clear, dim3((2 * D + 4 + 255) / 256), dim3(256), 0, stream, reinterpret_cast<uint32_t*>(c.mu), 2 * D + 4);
        // (a workgroup ends with two atomics per column, carried out one after the other: 123,457 x 37 with 64 rows each 0.062 ms, with 256
        // 0.022)
        const int g = std::max(1, std::min(N / (D <= 128 ? 256 : 64), 2048));
        if (D <= 128) hipLaunchKernelGGL(k_col_sum_narrow, dim3(g), dim3(256), 0, stream, points, N, D, c.mu, spread);
        else hipLaunchKernelGGL(k_col_sum, dim3(g), dim3(256), 0, stream, points, N, D, c.mu, spread);
        hipLaunchKernelGGL(k_col_mean, dim3(1), dim3(256), 0, stream, points, c.mu, spread, scale, D, 1.0f / (float)N);
    }
    const bool whole = (D & 3) == 0 && (reinterpret_cast<uintptr_t>(points) & 15) == 0;
    const int pitch = join_pitch(D);
#define RSFK_TO_JOIN(L)                                                                                                            \
    do {                                                                                                                           \
        c.n_parts = (int)std::min<size_t>(((size_t)N + 4 * (64 / L) - 1) / (4 * (64 / L)), kJoinMostGrid);                           \
        const dim3 grid((unsigned)c.n_parts);                                                                                      \
        if (whole) hipLaunchKernelGGL((k_to_join<L, true>), grid, dim3(256), 0, stream, points, c.rows, c.norms, c.errs, c.parts, c.mu, scale, N, D, pitch); \
        else hipLaunchKernelGGL((k_to_join<L, false>), grid, dim3(256), 0, stream, points, c.rows, c.norms, c.errs, c.parts, c.mu, scale, N, D, pitch); \
    } while (0)
    if (pitch <= 32) RSFK_TO_JOIN(8);
    else if (pitch <= 64) RSFK_TO_JOIN(16);
    else if (pitch <= 128) RSFK_TO_JOIN(32);
    else RSFK_TO_JOIN(64);
#undef RSFK_TO_JOIN
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
