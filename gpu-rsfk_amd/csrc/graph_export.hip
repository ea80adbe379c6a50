// Symmetrised K-NN graph in compressed-row form: row p holds every neighbour stored for p and every point that
// stores p as a neighbour, once, with the squared distance of the pair; columns ascend inside a row.  This is what
// consumers of the K-NN graph (t-SNE, UMAP, spectral methods) build first.  Replaces the three kernels the reference
// keeps commented out next to its spectral experiment (symmetric_knn_graph_edge_count / _offset / _add_edges,
// src/rsfk.cu:1229-1299: one thread per point, a serial prefix sum by a single thread, row order = arrival order of
// atomics).
//
// symmetrize_device: (1) the reversed graph by a counting sort in LDS (launch_reversed_graph, shared with the exploration:
// R(p) = the entries that hold p), (2) a wavefront per point drops from R(p) the points that p stores itself and counts
// what row p will hold, (3) prefix sum of the row lengths, (4) a wavefront per point gathers the union in LDS, ranks every
// column by counting the smaller ones and writes it to its place: no atomics on memory, no sort of the result (1M x 32:
// 3.71 -> 1.70 ms, 100,000 x 100: 1.46 -> 0.63).  Rows of more than 256 entries go to a workgroup each, which sorts them in LDS;
// those of points that more than some 4,000 others store (hubs) are gathered together and sorted by (row, column) in memory.
//
// The form below (symmetrize_flags) is for callers that cannot allocate, for small graphs, for inputs the builder of the
// reversed graph does not take and where there is no room for it: (1) a wavefront per point looks its own number up in the rows of its neighbours (coalesced row reads, four
// neighbours in flight) and counts, per point, the stored neighbours and the missing reverse edges; (2) prefix sum of
// the row lengths; (3) the edges are written to their rows: the stored ones at compacted positions, the added ones
// behind them in arrival order; (4) a segmented sort by column (rocPRIM) makes the rows independent of that order.
#include "forest.hpp"
#include "wave64.hpp"
#include "knn_list.hpp"
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_segmented_radix_sort.hpp>

namespace rsfk {

namespace {

constexpr unsigned char kNoEdge = 0, kMutual = 1, kOneWay = 2;

__device__ __forceinline__ bool usable(int c, int p, int N, int drop_self) { return c >= 0 && c < N && !(drop_self && c == p); }

// flag[p*K + k]: kNoEdge (empty slot, out of range, or a dropped self edge), kMutual (the neighbour stores p too),
// kOneWay (it does not: the reverse edge has to be added).  n_own[p] = stored edges of p, extra[p] (zero on entry) =
// reverse edges row p receives.
template <int SL>
__global__ __launch_bounds__(256) void k_sym_flags(const int* __restrict__ idx, int N, int K, int drop_self,
                                                   unsigned char* __restrict__ flag, int* __restrict__ n_own,
                                                   int* __restrict__ extra)
{
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (p >= N) return;
    int mine[SL];
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        const int k = lane + 64 * s;
        mine[s] = k < K ? idx[(size_t)p * K + k] : -1;
    }
    int own = 0;
    for (int k0 = 0; k0 < K; k0 += 4) {
        int pn[4];
        bool ok[4];
        int theirs[4][SL];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + u;
            int c = -1;
#pragma unroll
            for (int s = 0; s < SL; ++s)
                if ((k >> 6) == s) c = read_lane_i(mine[s], k & 63);
            pn[u] = c;
            ok[u] = k < K && usable(c, p, N, drop_self);
#pragma unroll
            for (int s = 0; s < SL; ++s) {
                const int kk = lane + 64 * s;
                theirs[u][s] = (ok[u] && kk < K) ? idx[(size_t)c * K + kk] : -1;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            bool hit = false;
#pragma unroll
            for (int s = 0; s < SL; ++s) hit |= theirs[u][s] == p;
            const bool mutual = ballot64(hit) != 0;
            if (k0 + u < K && lane == 0) {
                flag[(size_t)p * K + k0 + u] = !ok[u] ? kNoEdge : (mutual ? kMutual : kOneWay);
                if (ok[u] && !mutual) atomicAdd(&extra[pn[u]], 1);
            }
            own += ok[u] ? 1 : 0;
        }
    }
    if (lane == 0) n_own[p] = own;
}

// len[p] = length of row p; extra is set back to zero (it becomes the cursor of the added edges); len[N] = 0
__global__ __launch_bounds__(256) void k_sym_len(const int* __restrict__ n_own, int* __restrict__ extra, int N, int* __restrict__ len)
{
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p < N) { len[p] = n_own[p] + extra[p]; extra[p] = 0; }
    else if (p == N) len[p] = 0;
}

// Lane k of the wavefront of p writes the stored edge k to its compacted place in row p and, for a one-way edge, the
// reverse edge into the row of the neighbour behind that row's stored edges.
template <int SL>
__global__ __launch_bounds__(256) void k_sym_fill(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                  const unsigned char* __restrict__ flag, const int* __restrict__ n_own,
                                                  int* __restrict__ cursor, const int* __restrict__ indptr,
                                                  int* __restrict__ cols, float* __restrict__ vals)
{
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (p >= N) return;
    const int row0 = indptr[p];
    int before = 0;
#pragma unroll
    for (int s = 0; s < SL; ++s) {
        const int k = lane + 64 * s;
        const size_t e = (size_t)p * K + k;
        const int f = k < K ? flag[e] : kNoEdge;
        const uint64_t m = ballot64(f != kNoEdge);
        if (f != kNoEdge) {
            const int c = idx[e];
            const float d = dist ? dist[e] : 0.0f;
            const int at = row0 + before + __popcll(m & ((1ull << lane) - 1ull));
            cols[at] = c;
            vals[at] = d;
            if (f == kOneWay) {
                const int ra = indptr[c] + n_own[c] + atomicAdd(&cursor[c], 1);
                cols[ra] = p;
                vals[ra] = d;
            }
        }
        before += __popcll(m);
    }
}

int sym_launch_flags(const int* idx, int N, int K, int drop_self, unsigned char* flag, int* n_own, int* extra, hipStream_t stream)
{
    const dim3 grid((unsigned)((N + 3) / 4)), block(256);
    if (K <= 64) hipLaunchKernelGGL(k_sym_flags<1>, grid, block, 0, stream, idx, N, K, drop_self, flag, n_own, extra);
    else if (K <= 128) hipLaunchKernelGGL(k_sym_flags<2>, grid, block, 0, stream, idx, N, K, drop_self, flag, n_own, extra);
    else if (K <= 256) hipLaunchKernelGGL(k_sym_flags<4>, grid, block, 0, stream, idx, N, K, drop_self, flag, n_own, extra);
    else if (K <= 512) hipLaunchKernelGGL(k_sym_flags<8>, grid, block, 0, stream, idx, N, K, drop_self, flag, n_own, extra);
    else hipLaunchKernelGGL(k_sym_flags<16>, grid, block, 0, stream, idx, N, K, drop_self, flag, n_own, extra);
    RSFK_HIP(hipGetLastError());
    return 0;
}

int sym_launch_fill(const int* idx, const float* dist, int N, int K, const unsigned char* flag, const int* n_own, int* cursor,
                    const int* indptr, int* cols, float* vals, hipStream_t stream)
{
    const dim3 grid((unsigned)((N + 3) / 4)), block(256);
    if (K <= 64)
        hipLaunchKernelGGL(k_sym_fill<1>, grid, block, 0, stream, idx, dist, N, K, flag, n_own, cursor, indptr, cols, vals);
    else if (K <= 128)
        hipLaunchKernelGGL(k_sym_fill<2>, grid, block, 0, stream, idx, dist, N, K, flag, n_own, cursor, indptr, cols, vals);
    else if (K <= 256)
        hipLaunchKernelGGL(k_sym_fill<4>, grid, block, 0, stream, idx, dist, N, K, flag, n_own, cursor, indptr, cols, vals);
    else if (K <= 512)
        hipLaunchKernelGGL(k_sym_fill<8>, grid, block, 0, stream, idx, dist, N, K, flag, n_own, cursor, indptr, cols, vals);
    else
        hipLaunchKernelGGL(k_sym_fill<16>, grid, block, 0, stream, idx, dist, N, K, flag, n_own, cursor, indptr, cols, vals);
    RSFK_HIP(hipGetLastError());
    return 0;
}

struct Buf {
    void* p = nullptr;
    ~Buf() { if (p) ws_free(p); }
};

// ---- rows as unions --------------------------------------------------------------------------------------------------

constexpr int kUnionWave = 256;            // entries of a row a wavefront ranks (four per lane)
constexpr int kUnionBlock = 4096;          // candidates of a row a workgroup sorts in LDS

// Rows by the number of their entries and candidates (stored neighbours and reversed entries): a wavefront each up to
// kUnionWave entries, a workgroup each up to kUnionBlock candidates (`big`), the others (`hubs`) all together.
struct UnionCounters {
    int n_big;
    int pad;
    struct alignas(8) Hubs {
        unsigned entries;                  // of all hubs
        unsigned n;
    } hubs;
};
struct UnionLists {
    int* big;                              // points
    int2* hubs;                            // {point, entries of the hubs before it}
    UnionCounters* ctr;
};
// (a hub has more than kUnionBlock candidates, and all rows together 2 N K)
size_t most_hubs(size_t entries) { return 2 * entries / (size_t)kUnionBlock + 1; }

// The stored neighbours of p that are edges, in LDS and in order; returns their number.  (own: K ints of the wavefront.)
__device__ __forceinline__ int own_edges(const int* __restrict__ idx, int N, int K, int p, int drop_self, int* own)
{
    const int lane = threadIdx.x & 63;
    int n = 0;
    for (int k0 = 0; k0 < K; k0 += 64) {
        const int k = k0 + lane;
        const int c = k < K ? idx[(size_t)p * K + k] : -1;
        const bool ok = usable(c, p, N, drop_self);
        const uint64_t m = ballot64(ok);
        if (ok) own[n + mask_prefix(m)] = c;
        n += __popcll(m);
    }
    // padded to a multiple of four with what no point is
    if (lane < 4) own[n + lane] = -1;
    return n;
}

// Is c one of own[0..n)?  (every lane its own c)
__device__ __forceinline__ uint64_t in_own(const int* own, int n, int c)
{
    uint64_t m = 0;
    for (int j = 0; j < n; j += 4) {
        const int4 o = *reinterpret_cast<const int4*>(own + j);
        m |= mask_eq_i(o.x, c) | mask_eq_i(o.y, c) | mask_eq_i(o.z, c) | mask_eq_i(o.w, c);
    }
    return m;
}

// len[p] = entries of row p; len[N] = 0.
__global__ __launch_bounds__(256) void k_union_len(const int* __restrict__ idx, int N, int K, int drop_self, const int* __restrict__ offs,
                                                   const int* __restrict__ rev, uint32_t div_m, int div_s, int own_ints,
                                                   int* __restrict__ len, UnionLists L)
{
    extern __shared__ __align__(16) int union_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = (int)blockIdx.x * 4 + wave;
    if (p >= N) {
        if (p == N && lane == 0) len[N] = 0;
        return;
    }
    int* own = union_lds + wave * own_ints;
    const int r0 = offs[p], r1 = offs[p + 1];
    const int e0 = r0 + lane < r1 ? rev[r0 + lane] : -1;
    const int n = own_edges(idx, N, K, p, drop_self, own);
    wave_lds_sync();
    int total = n;
    auto count = [&](int e) {
        const int c = (int)(((uint64_t)(uint32_t)e * div_m) >> div_s);
        const bool ok = e >= 0 && !(drop_self && c == p);
        total += __popcll(ballot64(ok) & ~in_own(own, n, c));
    };
    if (r0 < r1) count(e0);
    // (eight loads at a time: R(p) of a hub is long)
    for (int r = r0 + 64; r < r1; r += 512) {
        int e[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) e[u] = r + 64 * u + lane < r1 ? rev[r + 64 * u + lane] : -1;
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (r + 64 * u < r1) count(e[u]);
    }
    if (lane == 0) {
        len[p] = total;
        if (n + (r1 - r0) > kUnionBlock) {
            const unsigned long long was = atomicAdd(reinterpret_cast<unsigned long long*>(&L.ctr->hubs), (unsigned)total | (1ull << 32));
            L.hubs[was >> 32] = make_int2(p, (int)(unsigned)was);
        } else if (total > kUnionWave) {
            L.big[atomicAdd(&L.ctr->n_big, 1)] = p;
        }
    }
}

// Entries 64 S and fewer: lane l has the entries l, l + 64, ..; the place of an entry is the number of smaller columns.
template <int S>
__device__ __forceinline__ void rank_and_store(const int* key, const int* entry, int n, const float* __restrict__ dist,
                                               int* __restrict__ cols, float* __restrict__ vals)
{
    const int lane = threadIdx.x & 63;
    int k[S], rank[S];
    float v[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        const int i = lane + 64 * s;
        k[s] = i < n ? key[i] : 0x7fffffff;
        v[s] = i < n && dist ? dist[entry[i]] : 0.0f;
        rank[s] = 0;
    }
    for (int j = 0; j < n; j += 4) {
        const int4 o = *reinterpret_cast<const int4*>(key + j);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            rank[s] += o.x < k[s] ? 1 : 0;
            rank[s] += o.y < k[s] ? 1 : 0;
            rank[s] += o.z < k[s] ? 1 : 0;
            rank[s] += o.w < k[s] ? 1 : 0;
        }
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
        if (lane + 64 * s < n) {
            cols[rank[s]] = k[s];
            vals[rank[s]] = v[s];
        }
}

// Row p from the stored neighbours and the reversed entries that are not among them (a wavefront each).  What bounds it: the
// gather of the reversed entries' distances (one 4-byte word per added edge) and the comparisons (two instructions per
// column and lane).
__global__ __launch_bounds__(256) void k_union_fill(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                    int drop_self, const int* __restrict__ offs, const int* __restrict__ rev,
                                                    uint32_t div_m, int div_s, int own_ints, const int* __restrict__ indptr,
                                                    long long cap, int* __restrict__ cols, float* __restrict__ vals)
{
    extern __shared__ __align__(16) int union_lds[];
    if (indptr[N] > cap) return;                                        // (the host reports)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = (int)blockIdx.x * 4 + wave;
    if (p >= N) return;
    const int row0 = indptr[p], n_row = indptr[p + 1] - row0;
    if (n_row == 0 || n_row > kUnionWave) return;
    int* own = union_lds + wave * (own_ints + 2 * (kUnionWave + 4));
    int* key = own + own_ints;
    int* entry = key + kUnionWave + 4;
    const int r0 = offs[p], r1 = offs[p + 1];
    const int e0 = r0 + lane < r1 ? rev[r0 + lane] : -1;
    int n = 0;
    for (int k0 = 0; k0 < K; k0 += 64) {
        const int k = k0 + lane;
        const int c = k < K ? idx[(size_t)p * K + k] : -1;
        const bool ok = usable(c, p, N, drop_self);
        const uint64_t m = ballot64(ok);
        if (ok) {
            const int at = n + mask_prefix(m);
            own[at] = c;
            key[at] = c;
            entry[at] = p * K + k;
        }
        n += __popcll(m);
    }
    if (lane < 4) own[n + lane] = -1;
    wave_lds_sync();
    int total = n;
    for (int r = r0; r < r1; r += 64) {
        const int e = r == r0 ? e0 : (r + lane < r1 ? rev[r + lane] : -1);
        const int c = (int)(((uint64_t)(uint32_t)e * div_m) >> div_s);
        const bool ok = e >= 0 && !(drop_self && c == p);
        const uint64_t m = ballot64(ok) & ~in_own(own, n, c);
        if (lane_bit(m)) {
            const int at = total + mask_prefix(m);
            key[at] = c;
            entry[at] = e;
        }
        total += __popcll(m);
    }
    if (lane < 4) key[total + lane] = 0x7fffffff;                        // (counts for nobody)
    wave_lds_sync();
    if (n_row <= 64) rank_and_store<1>(key, entry, n_row, dist, cols + row0, vals + row0);
    else if (n_row <= 128) rank_and_store<2>(key, entry, n_row, dist, cols + row0, vals + row0);
    else rank_and_store<4>(key, entry, n_row, dist, cols + row0, vals + row0);
}

// Rows of more than kUnionWave entries: all candidates (column << 32 | entry number, stored neighbours before reversed entries
// of the same column) sorted in LDS by a workgroup, of equal columns the first one kept.
__global__ __launch_bounds__(256) void k_union_fill_big(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                        int drop_self, const int* __restrict__ offs, const int* __restrict__ rev,
                                                        uint32_t div_m, int div_s, const int* __restrict__ indptr,
                                                        UnionLists L, long long cap, int* __restrict__ cols,
                                                        float* __restrict__ vals)
{
    __shared__ unsigned long long a[kUnionBlock];
    __shared__ int n_s, wave_n[4];
    if (indptr[N] > cap) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_big = L.ctr->n_big;
    constexpr unsigned long long kNone = ~0ull;
    for (int b = blockIdx.x; b < n_big; b += gridDim.x) {
        const int p = L.big[b];
        __syncthreads();
        if (tid == 0) n_s = 0;
        __syncthreads();
        for (int k = tid; k < K; k += 256) {
            const int c = idx[(size_t)p * K + k];
            if (usable(c, p, N, drop_self)) a[atomicAdd(&n_s, 1)] = ((unsigned long long)(unsigned)c << 32) | (unsigned)(p * K + k);
        }
        const int r0 = offs[p], r1 = offs[p + 1];
        for (int r = r0 + tid; r < r1; r += 256) {
            const int e = rev[r];
            const int c = (int)(((uint64_t)(uint32_t)e * div_m) >> div_s);
            if (!(drop_self && c == p)) a[atomicAdd(&n_s, 1)] = ((unsigned long long)(unsigned)c << 32) | 0x80000000ull | (unsigned)e;
        }
        __syncthreads();
        const int n = n_s;
        int m = 1;
        while (m < n) m <<= 1;
        for (int i = n + tid; i < m; i += 256) a[i] = kNone;
        for (int size = 2; size <= m; size <<= 1)
            for (int step = size >> 1; step > 0; step >>= 1) {
                __syncthreads();
                for (int i = tid; i < m / 2; i += 256) {
                    const int lo = 2 * i - (i & (step - 1)), hi = lo + step;
                    const bool up = (lo & size) == 0;
                    const unsigned long long x = a[lo], y = a[hi];
                    if ((x > y) == up) { a[lo] = y; a[hi] = x; }
                }
            }
        __syncthreads();
        int* out_c = cols + indptr[p];
        float* out_v = vals + indptr[p];
        int done = 0;
        for (int i0 = 0; i0 < n; i0 += 256) {
            const int i = i0 + tid;
            const unsigned long long x = i < n ? a[i] : kNone;
            const bool keep = i < n && (i == 0 || (unsigned)(a[i - 1] >> 32) != (unsigned)(x >> 32));
            const uint64_t mk = ballot64(keep);
            if (lane == 0) wave_n[wave] = __popcll(mk);
            __syncthreads();
            int at = done + mask_prefix(mk);
            for (int w = 0; w < 4; ++w) {
                if (w < wave) at += wave_n[w];
                done += wave_n[w];
            }
            if (keep) {
                out_c[at] = (int)(unsigned)(x >> 32);
                out_v[at] = dist ? dist[(unsigned)x & 0x7fffffffu] : 0.0f;
            }
            __syncthreads();
        }
    }
}

__global__ void k_union_zero(UnionCounters* ctr)
{
    *ctr = UnionCounters();
}

// Hubs (a row of blockIdx.x each, blockIdx.y: a share of R(p)): the entries of their rows in any order, key = number of the hub
// << col_bits | column, of equal columns the stored neighbour.  cursor (zero on entry) counts them.  A row of any length is too
// long for the LDS of one workgroup, but the hubs' rows together are a small part of the graph, so that sorting them costs
// little beside the rest: 1M x 32 with one hub of 10,000 entries 1.76 ms (3.87 with all rows in the other form), with 20 hubs
// of 300,000 each 14.5 (72), 100,000 x 16 with one hub of 6,000 0.198 (0.416).
__global__ __launch_bounds__(256) void k_hub_gather(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                    int drop_self, const int* __restrict__ offs, const int* __restrict__ rev,
                                                    uint32_t div_m, int div_s, int own_ints, const int2* __restrict__ hubs, int col_bits,
                                                    int* __restrict__ cursor, unsigned long long* __restrict__ keys,
                                                    float* __restrict__ vals)
{
    extern __shared__ __align__(16) int union_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.x, p = hubs[h].x, first = hubs[h].y;
    int* own = union_lds + wave * own_ints;
    const int n = own_edges(idx, N, K, p, drop_self, own);
    wave_lds_sync();
    const unsigned long long row = (unsigned long long)(unsigned)h << col_bits;
    auto put = [&](bool keep, int c, int e) {
        const uint64_t m = ballot64(keep);
        if (m == 0) return;
        int at = lane == 0 ? atomicAdd(&cursor[h], __popcll(m)) : 0;
        at = first + __builtin_amdgcn_readfirstlane(at) + mask_prefix(m);
        if (keep) {
            keys[at] = row | (unsigned)c;
            vals[at] = dist ? dist[e] : 0.0f;
        }
    };
    if (blockIdx.y == 0 && wave == 0)
        for (int k0 = 0; k0 < K; k0 += 64) {
            const int k = k0 + lane, e = p * K + k;
            const int c = k < K ? idx[e] : -1;
            put(usable(c, p, N, drop_self), c, e);
        }
    const int r1 = offs[p + 1], step = (int)gridDim.y * 256;
    for (int r = offs[p] + ((int)blockIdx.y * 4 + wave) * 64; r < r1; r += step) {
        const int e = r + lane < r1 ? rev[r + lane] : -1;
        const int c = (int)(((uint64_t)(uint32_t)e * div_m) >> div_s);
        const bool ok = e >= 0 && !(drop_self && c == p);
        put(lane_bit(ballot64(ok) & ~in_own(own, n, c)), c, e);
    }
}

// The sorted entries of the hubs to their rows.
__global__ __launch_bounds__(256) void k_hub_store(const unsigned long long* __restrict__ keys, const float* __restrict__ sorted, unsigned n,
                                                   const int2* __restrict__ hubs, int col_bits, const int* __restrict__ indptr,
                                                   int* __restrict__ cols, float* __restrict__ vals)
{
    const unsigned i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const unsigned long long key = keys[i];
    const int2 hub = hubs[key >> col_bits];
    const int at = indptr[hub.x] + (int)(i - (unsigned)hub.y);
    cols[at] = (int)(key & ((1ull << col_bits) - 1ull));
    vals[at] = sorted[i];
}

__global__ __launch_bounds__(256) void k_zero_counters(int* __restrict__ v, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) v[i] = 0;
}

struct RevGuard {
    ExploreWorkspace* w = nullptr;
    ~RevGuard() { explore_ws_free(w); }
};

// Where the rows go: arrays of the caller with room for `cap` entries (both null: only the row offsets and the count are wanted),
// or (make) arrays of the size of the graph, made here once that is known.
struct GraphOut {
    int* cols = nullptr;
    float* vals = nullptr;
    long long cap = 0;
    bool make = false;
    Buf c, v;
    // nnz is known: 0, or nonzero with the reason when the arrays cannot take it
    int room(long long nnz)
    {
        RSFK_CHECK(nnz <= cap, "graph export: the output arrays are too small for the graph");
        if (!make) return 0;
        if (ws_alloc(&c.p, sizeof(int) * (size_t)nnz) || ws_alloc(&v.p, sizeof(float) * (size_t)nnz)) return 1;
        cols = static_cast<int*>(c.p);
        vals = static_cast<float*>(v.p);
        return 0;
    }
    bool wanted() const { return make || cols != nullptr; }
};

int symmetrize_flags(const int* d_idx, const float* d_dist, int N, int K, int drop_self, int* d_indptr, GraphOut& out,
                     long long* nnz, hipStream_t stream);

int symmetrize(const int* d_idx, const float* d_dist, int N, int K, int drop_self, int* d_indptr, GraphOut& out, long long* nnz,
               hipStream_t stream)
{
    RSFK_CHECK(N >= 1 && K >= 1 && K <= kMaxK, "graph export: N must be positive and K in 1..1024");
    RSFK_CHECK((long long)N * K < (1ll << 30), "graph export: N * K of 2^30 and more is not supported");
    RSFK_CHECK(d_idx && d_indptr && nnz, "graph export: null argument");
    // Up to about 2,800 points the library's sort takes few launches and the other form fewer in all (2,000 x 32: 0.057 against
    // 0.059 ms, 2,000 x 128: 0.102 against 0.141; 2,500 x 8: 0.049 against 0.048); from there on it takes more (3,000 x 8: 0.076
    // against 0.050, 3,000 x 90: 0.118 against 0.101).  RSFK_GRAPH_FLAGS=1 / 0 says which form (the results are the same).
    const char* form = std::getenv("RSFK_GRAPH_FLAGS");
    if (!explore_ws_takes(N, K) || (form && *form ? form[0] == '1' : N < 2800))
        return symmetrize_flags(d_idx, d_dist, N, K, drop_self, d_indptr, out, nnz, stream);
    RevGuard rg;
    Buf len, big, hubs, ctr;
    // the reversed graph takes 12 bytes per entry (20 from 2^26 entries on), the other form one
    if (explore_ws_alloc(&rg.w, N, K, false, true))
        return symmetrize_flags(d_idx, d_dist, N, K, drop_self, d_indptr, out, nnz, stream);
    if (ws_alloc(&len.p, sizeof(int) * ((size_t)N + 1)) || ws_alloc(&big.p, sizeof(int) * (size_t)N) ||
        ws_alloc(&hubs.p, sizeof(int2) * most_hubs((size_t)N * (size_t)K)) || ws_alloc(&ctr.p, sizeof(UnionCounters)))
        return 1;
    const UnionLists L = {static_cast<int*>(big.p), static_cast<int2*>(hubs.p), static_cast<UnionCounters*>(ctr.p)};
    hipLaunchKernelGGL(k_union_zero, dim3(1), dim3(1), 0, stream, L.ctr);
    if (launch_reversed_graph(rg.w, d_idx, N, K, stream)) return 1;
    const int* offs = explore_ws_offs(rg.w);
    const int* rev = explore_ws_rev(rg.w);
    // e / K for 0 <= e < 2^30
    int l = 0;
    while ((1 << l) < K) ++l;
    const int div_s = 31 + l;
    const uint32_t div_m = (uint32_t)((((uint64_t)1 << div_s) + (uint64_t)K - 1) / (uint64_t)K);
    const int own_ints = (K + 4 + 3) & ~3;
    hipLaunchKernelGGL(k_union_len, dim3((unsigned)(N / 4 + 1)), dim3(256), (size_t)4 * own_ints * sizeof(int), stream, d_idx, N, K,
                       drop_self, offs, rev, div_m, div_s, own_ints, static_cast<int*>(len.p), L);
    RSFK_HIP(hipGetLastError());
    size_t tmp_bytes = 0;
    RSFK_HIP(rocprim::exclusive_scan(nullptr, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                     rocprim::plus<int>(), stream));
    Buf tmp;
    if (ws_alloc(&tmp.p, tmp_bytes ? tmp_bytes : 256)) return 1;
    RSFK_HIP(rocprim::exclusive_scan(tmp.p, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                     rocprim::plus<int>(), stream));
    const auto fill = [&]() -> int {
        const size_t lds = (size_t)4 * (own_ints + 2 * (kUnionWave + 4)) * sizeof(int);
        hipLaunchKernelGGL(k_union_fill, dim3((unsigned)((N + 3) / 4)), dim3(256), lds, stream, d_idx, d_dist, N, K, drop_self, offs, rev,
                           div_m, div_s, own_ints, d_indptr, out.cap, out.cols, out.vals);
        hipLaunchKernelGGL(k_union_fill_big, dim3(256), dim3(256), 0, stream, d_idx, d_dist, N, K, drop_self, offs, rev, div_m, div_s,
                           d_indptr, L, out.cap, out.cols, out.vals);
        RSFK_HIP(hipGetLastError());
        return 0;
    };
    // one trip to the host, for arrays of the caller after everything has been queued
    if (out.cols && fill()) return 1;
    int word[3] = {0, 0, 0};                                     // entries, entries of the hubs, hubs
    if (fetch_words(d_indptr + N, 1, reinterpret_cast<const int*>(&L.ctr->hubs), 2, word, stream)) return 1;
    *nnz = word[0];
    if (!out.wanted() || *nnz == 0) return 0;
    const int n_hubs = word[2];
    const size_t n_entries = (size_t)(unsigned)word[1];
    Buf cursor, keys[2], sorted[2];
    if (n_hubs > 0) {
        // 24 bytes per entry of a hub; the other form does without them
        if (ws_try_alloc(&cursor.p, sizeof(int) * (size_t)n_hubs)) cursor.p = nullptr;
        bool have = cursor.p != nullptr;
        for (int i = 0; i < 2 && have; ++i)
            have = ws_try_alloc(&keys[i].p, sizeof(unsigned long long) * n_entries) == 0 && ws_try_alloc(&sorted[i].p, sizeof(float) * n_entries) == 0;
        if (!have) return symmetrize_flags(d_idx, d_dist, N, K, drop_self, d_indptr, out, nnz, stream);
    }
    if (out.room(*nnz)) return 1;
    if (out.make && fill()) return 1;
    if (n_hubs > 0) {
        int col_bits = 1, hub_bits = 1;
        while ((1ll << col_bits) < (long long)N) ++col_bits;
        while ((1ll << hub_bits) < (long long)n_hubs) ++hub_bits;
        unsigned long long* key[2] = {static_cast<unsigned long long*>(keys[0].p), static_cast<unsigned long long*>(keys[1].p)};
        float* val[2] = {static_cast<float*>(sorted[0].p), static_cast<float*>(sorted[1].p)};
        hipLaunchKernelGGL(k_zero_counters, dim3((unsigned)((n_hubs + 255) / 256)), dim3(256), 0, stream, static_cast<int*>(cursor.p), n_hubs);
        // about 2,000 workgroups over all hubs, each with 1,024 entries of R(p) or more
        const size_t mean = n_entries / (size_t)n_hubs;
        const unsigned shares = (unsigned)std::max<size_t>(1, std::min<size_t>(mean / 1024, (size_t)(2048 / std::min(n_hubs, 2048))));
        hipLaunchKernelGGL(k_hub_gather, dim3((unsigned)n_hubs, shares), dim3(256), (size_t)4 * own_ints * sizeof(int), stream, d_idx, d_dist,
                           N, K, drop_self, offs, rev, div_m, div_s, own_ints, L.hubs, col_bits, static_cast<int*>(cursor.p), key[0], val[0]);
        RSFK_HIP(hipGetLastError());
        size_t sort_bytes = 0;
        RSFK_HIP(rocprim::radix_sort_pairs(nullptr, sort_bytes, key[0], key[1], val[0], val[1], n_entries, 0, (unsigned)(col_bits + hub_bits), stream));
        Buf tmp_sort;
        if (ws_alloc(&tmp_sort.p, sort_bytes ? sort_bytes : 256)) return 1;
        RSFK_HIP(rocprim::radix_sort_pairs(tmp_sort.p, sort_bytes, key[0], key[1], val[0], val[1], n_entries, 0, (unsigned)(col_bits + hub_bits), stream));
        hipLaunchKernelGGL(k_hub_store, dim3((unsigned)((n_entries + 255) / 256)), dim3(256), 0, stream, key[1], val[1], (unsigned)n_entries,
                           L.hubs, col_bits, d_indptr, out.cols, out.vals);
        RSFK_HIP(hipGetLastError());
        RSFK_HIP(hipStreamSynchronize(stream));
        return 0;
    }
    if (out.make) RSFK_HIP(hipStreamSynchronize(stream));        // (the working memory goes back to the pool)
    return 0;
}

int symmetrize_flags(const int* d_idx, const float* d_dist, int N, int K, int drop_self, int* d_indptr, GraphOut& out,
                     long long* nnz, hipStream_t stream)
{
    Buf flag, own, extra, len;
    if (ws_alloc(&flag.p, (size_t)N * K) || ws_alloc(&own.p, sizeof(int) * (size_t)N) ||
        ws_alloc(&extra.p, sizeof(int) * (size_t)N) || ws_alloc(&len.p, sizeof(int) * ((size_t)N + 1)))
        return 1;
    int* n_own = static_cast<int*>(own.p);
    int* ext = static_cast<int*>(extra.p);
    RSFK_HIP(hipMemsetAsync(ext, 0, sizeof(int) * (size_t)N, stream));
    if (sym_launch_flags(d_idx, N, K, drop_self, static_cast<unsigned char*>(flag.p), n_own, ext, stream)) return 1;
    hipLaunchKernelGGL(k_sym_len, dim3((unsigned)(N / 256 + 1)), dim3(256), 0, stream, n_own, ext, N, static_cast<int*>(len.p));
    RSFK_HIP(hipGetLastError());
    size_t tmp_bytes = 0;
    RSFK_HIP(rocprim::exclusive_scan(nullptr, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                     rocprim::plus<int>(), stream));
    {
        Buf tmp;
        if (ws_alloc(&tmp.p, tmp_bytes ? tmp_bytes : 256)) return 1;
        RSFK_HIP(rocprim::exclusive_scan(tmp.p, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                         rocprim::plus<int>(), stream));
        int total = 0;
        if (fetch_words(d_indptr + N, 1, &total, stream)) return 1;
        *nnz = total;
    }
    if (!out.wanted() || *nnz == 0) return 0;
    if (out.room(*nnz)) return 1;
    int* d_cols = out.cols;
    float* d_vals = out.vals;
    const size_t n = (size_t)*nnz;
    Buf cols, vals;
    if (ws_alloc(&cols.p, sizeof(int) * n) || ws_alloc(&vals.p, sizeof(float) * n)) return 1;
    if (sym_launch_fill(d_idx, d_dist, N, K, static_cast<unsigned char*>(flag.p), n_own, ext, d_indptr,
                        static_cast<int*>(cols.p), static_cast<float*>(vals.p), stream))
        return 1;
    int bits = 1;
    while (bits < 31 && (1ll << bits) < (long long)N) ++bits;          // columns are below N
    size_t sort_bytes = 0;
    RSFK_HIP(rocprim::segmented_radix_sort_pairs(nullptr, sort_bytes, static_cast<int*>(cols.p), d_cols,
                                                 static_cast<float*>(vals.p), d_vals, (unsigned)n, (unsigned)N, d_indptr,
                                                 d_indptr + 1, 0, (unsigned)bits, stream));
    Buf tmp;
    if (ws_alloc(&tmp.p, sort_bytes ? sort_bytes : 256)) return 1;
    RSFK_HIP(rocprim::segmented_radix_sort_pairs(tmp.p, sort_bytes, static_cast<int*>(cols.p), d_cols,
                                                 static_cast<float*>(vals.p), d_vals, (unsigned)n, (unsigned)N, d_indptr,
                                                 d_indptr + 1, 0, (unsigned)bits, stream));
    RSFK_HIP(hipStreamSynchronize(stream));
    return 0;
}

}  // namespace

// d_idx / d_dist: N x K (d_dist may be null: the values are then zero).  d_indptr: N + 1 ints.  d_cols / d_vals: room for
// `cap` entries, or both null to obtain only d_indptr and *nnz.  Entries that are negative or >= N are no edges;
// drop_self removes p from its own row.  A row must not hold a point twice.
int symmetrize_device(const int* d_idx, const float* d_dist, int N, int K, int drop_self, int* d_indptr, int* d_cols,
                      float* d_vals, long long cap, long long* nnz, hipStream_t stream)
{
    RSFK_CHECK((d_cols == nullptr) == (d_vals == nullptr), "graph export: indices and data go together");
    GraphOut out;
    out.cols = d_cols;
    out.vals = d_vals;
    out.cap = cap;
    return symmetrize(d_idx, d_dist, N, K, drop_self, d_indptr, out, nnz, stream);
}

// ---------------------------------------------------------------------------------------------------------------------
// The count-only call (row lengths, d_indptr and the number of entries) for callers that cannot allocate device memory:
// tight serving loops, harnesses that forbid hipMalloc, code that records a HIP graph.  With nnz == nullptr the call
// only enqueues kernels (the count is left in d_indptr[N] on the device); with nnz != nullptr it also copies the
// count to the host and synchronises the stream, which a stream under capture refuses.  Its working memory -- the edge
// flags, the three per-point counters and the temporary storage of the prefix sum, which symmetrize_device takes from
// the workspace pool -- lives in a file-scope device array of fixed size.  Every GPU the library runs on holds its
// own copy of that array until the process ends; its address on a device is looked up once per device and kept.
// All calls on one GPU share the array: calls that overlap on one GPU (two streams, two threads) race.
// ---------------------------------------------------------------------------------------------------------------------
namespace {

constexpr int kNaMaxPoints = 1 << 20;                     // N
constexpr long long kNaMaxSlots = 1ll << 25;              // N * K
constexpr size_t kNaScanBytes = (size_t)1 << 20;          // temporary storage of the prefix sum over N + 1 row lengths
constexpr size_t kNaCounterBytes = ((sizeof(int) * ((size_t)kNaMaxPoints + 1) + 255) / 256) * 256;
constexpr size_t kNaFlagOff = 0;
constexpr size_t kNaOwnOff = kNaFlagOff + (size_t)kNaMaxSlots;
constexpr size_t kNaExtraOff = kNaOwnOff + kNaCounterBytes;
constexpr size_t kNaLenOff = kNaExtraOff + kNaCounterBytes;
constexpr size_t kNaScanOff = kNaLenOff + kNaCounterBytes;
constexpr size_t kNaBytes = kNaScanOff + kNaScanBytes;    // 32 MiB + 3 x 4 MiB + 1 MiB

static __device__ __align__(256) unsigned char scratch[kNaBytes];

constexpr int kNaMaxDevices = 64;
unsigned char* g_scratch_ptr[kNaMaxDevices];              // device address of `scratch` on each device, once known
std::mutex g_scratch_mutex;

// The device address of the array on the current device.  The array's name is only a host-side handle.
int scratch_on_current_device(unsigned char** out)
{
    int dev = -1;
    RSFK_HIP(hipGetDevice(&dev));
    RSFK_CHECK(dev >= 0 && dev < kNaMaxDevices, "graph export: device number out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        RSFK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        RSFK_CHECK(p != nullptr, "graph export: no device address for the working memory");
        g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch_ptr[dev];
    return 0;
}

}  // namespace

int symmetrize_count_noalloc(const int* d_idx, int N, int K, int drop_self, int* d_indptr, long long* nnz, hipStream_t stream)
{
    RSFK_CHECK(d_idx && d_indptr, "graph export: null argument");
    RSFK_CHECK(N >= 1 && K >= 1 && K <= kMaxK, "graph export: N must be positive and K in 1..1024");
    RSFK_CHECK(N <= kNaMaxPoints && (long long)N * K <= kNaMaxSlots,
               "graph export without allocation: at most 2^20 points and 2^25 neighbour slots (N * K)");
    unsigned char* base = nullptr;
    if (scratch_on_current_device(&base)) return 1;
    unsigned char* flag = base + kNaFlagOff;
    int* n_own = reinterpret_cast<int*>(base + kNaOwnOff);
    int* ext = reinterpret_cast<int*>(base + kNaExtraOff);
    int* len = reinterpret_cast<int*>(base + kNaLenOff);
    void* scan_tmp = base + kNaScanOff;
    size_t tmp_bytes = 0;
    RSFK_HIP(rocprim::exclusive_scan(nullptr, tmp_bytes, len, d_indptr, 0, (size_t)N + 1, rocprim::plus<int>(), stream));
    RSFK_CHECK(tmp_bytes <= kNaScanBytes, "graph export without allocation: the prefix sum needs more temporary storage than reserved");
    // the counters of the reverse edges must start at zero; the array keeps the previous call's contents
    hipLaunchKernelGGL(k_zero_counters, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, stream, ext, N);
    RSFK_HIP(hipGetLastError());
    if (sym_launch_flags(d_idx, N, K, drop_self, flag, n_own, ext, stream)) return 1;
    hipLaunchKernelGGL(k_sym_len, dim3((unsigned)(N / 256 + 1)), dim3(256), 0, stream, n_own, ext, N, len);
    RSFK_HIP(hipGetLastError());
    RSFK_HIP(rocprim::exclusive_scan(scan_tmp, tmp_bytes, len, d_indptr, 0, (size_t)N + 1, rocprim::plus<int>(), stream));
    if (nnz == nullptr) return 0;                       // the count stays in d_indptr[N]; nothing but kernels was queued
    int total = 0;
    RSFK_HIP(hipMemcpyAsync(&total, d_indptr + N, sizeof(int), hipMemcpyDeviceToHost, stream));
    RSFK_HIP(hipStreamSynchronize(stream));
    *nnz = total;
    return 0;
}

int symmetrize_host(const int* idx, const float* dist, int N, int K, int drop_self, int* indptr, int* cols, float* vals,
                    long long cap, long long* nnz)
{
    RSFK_CHECK(N >= 1 && K >= 1, "graph export: N and K must be positive");
    RSFK_CHECK(idx && indptr && nnz, "graph export: null argument");
    RSFK_CHECK((cols == nullptr) == (vals == nullptr), "graph export: indices and data go together");
    HostStage stage;
    Buf di, dd, dp;
    const size_t nk = (size_t)N * K;
    if (ws_alloc(&di.p, nk * sizeof(int)) || ws_alloc(&dp.p, ((size_t)N + 1) * sizeof(int))) return 1;
    if (dist && ws_alloc(&dd.p, nk * sizeof(float))) return 1;
    GraphOut rows;
    rows.make = cols != nullptr && cap > 0;
    rows.cap = cap;
    const HostArray in[] = {{di.p, const_cast<int*>(idx), nk * sizeof(int)}, {dd.p, const_cast<float*>(dist), nk * sizeof(float)}};
    if (stage.to_device(in, dist ? 2 : 1, nullptr)) return 1;
    const int rc = symmetrize(static_cast<const int*>(di.p), static_cast<const float*>(dd.p), N, K, drop_self,
                              static_cast<int*>(dp.p), rows, nnz, nullptr);
    if (rc) return rc;
    const HostArray out[] = {{dp.p, indptr, ((size_t)N + 1) * sizeof(int)}, {rows.cols, cols, (size_t)*nnz * sizeof(int)},
                             {rows.vals, vals, (size_t)*nnz * sizeof(float)}};
    return copy_to_host(out, rows.cols ? 3 : 1, nullptr);
}

}  // namespace rsfk
