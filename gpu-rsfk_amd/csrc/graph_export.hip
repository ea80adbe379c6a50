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
// reverse edges row p receives.  One wavefront per point, from point `first` on.
template <int SL>
__global__ __launch_bounds__(256) void k_sym_flags(const int* __restrict__ idx, int first, int N, int K, int drop_self,
                                                   unsigned char* __restrict__ flag, int* __restrict__ n_own,
                                                   int* __restrict__ extra)
{
    const int lane = threadIdx.x & 63;
    const int p = first + blockIdx.x * 4 + (threadIdx.x >> 6);
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
__global__ __launch_bounds__(256) void k_sym_fill(const int* __restrict__ idx, const float* __restrict__ dist, int first, int N, int K,
                                                  const unsigned char* __restrict__ flag, const int* __restrict__ n_own,
                                                  int* __restrict__ cursor, const int* __restrict__ indptr,
                                                  int* __restrict__ cols, float* __restrict__ vals)
{
    const int lane = threadIdx.x & 63;
    const int p = first + blockIdx.x * 4 + (threadIdx.x >> 6);
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
    for (int first = 0; first < N; first += std::min(kMostRows, N - first)) {
        const dim3 grid((unsigned)((std::min(kMostRows, N - first) + 3) / 4)), block(256);
        if (K <= 64) hipLaunchKernelGGL(k_sym_flags<1>, grid, block, 0, stream, idx, first, N, K, drop_self, flag, n_own, extra);
        else if (K <= 128) hipLaunchKernelGGL(k_sym_flags<2>, grid, block, 0, stream, idx, first, N, K, drop_self, flag, n_own, extra);
        else if (K <= 256) hipLaunchKernelGGL(k_sym_flags<4>, grid, block, 0, stream, idx, first, N, K, drop_self, flag, n_own, extra);
        else if (K <= 512) hipLaunchKernelGGL(k_sym_flags<8>, grid, block, 0, stream, idx, first, N, K, drop_self, flag, n_own, extra);
        else hipLaunchKernelGGL(k_sym_flags<16>, grid, block, 0, stream, idx, first, N, K, drop_self, flag, n_own, extra);
    }
    RSFK_HIP(hipGetLastError());
    return 0;
}

int sym_launch_fill(const int* idx, const float* dist, int N, int K, const unsigned char* flag, const int* n_own, int* cursor,
                    const int* indptr, int* cols, float* vals, hipStream_t stream)
{
    for (int first = 0; first < N; first += std::min(kMostRows, N - first)) {
        const dim3 grid((unsigned)((std::min(kMostRows, N - first) + 3) / 4)), block(256);
        if (K <= 64)
            hipLaunchKernelGGL(k_sym_fill<1>, grid, block, 0, stream, idx, dist, first, N, K, flag, n_own, cursor, indptr, cols, vals);
        else if (K <= 128)
            hipLaunchKernelGGL(k_sym_fill<2>, grid, block, 0, stream, idx, dist, first, N, K, flag, n_own, cursor, indptr, cols, vals);
        else if (K <= 256)
            hipLaunchKernelGGL(k_sym_fill<4>, grid, block, 0, stream, idx, dist, first, N, K, flag, n_own, cursor, indptr, cols, vals);
        else if (K <= 512)
            hipLaunchKernelGGL(k_sym_fill<8>, grid, block, 0, stream, idx, dist, first, N, K, flag, n_own, cursor, indptr, cols, vals);
        else
            hipLaunchKernelGGL(k_sym_fill<16>, grid, block, 0, stream, idx, dist, first, N, K, flag, n_own, cursor, indptr, cols, vals);
    }
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

// A wavefront takes PTS consecutive points, whose stored neighbours and reversed entries follow each other in memory: what such a
// wavefront waits for is its trips (offsets, then rows and reversed entries, then distances), not bytes or instructions (1M x 32, one
// point per wavefront: lengths 0.30 ms, rows 0.53; four: 0.18 and 0.32.  With 4 or 16 slots per neighbour the lengths take 0.23 and 0.26).
// Few points do not fill the device, and a wavefront's work counts (lengths and rows in us with one, two and four points: 3,001 x 32 9.2,
// 13.8, 17.5; 14,009 x 32 16.6, 16.8, 21.0; 60,013 x 32 46.9, 40.6, 41.3; 6,007 x 16 8.2, 8.4, 10.7; 20,011 x 16 17.1, 14.5, 13.8; 14,009 x 5
// 12.3, 9.8, 9.6; 30,011 x 48 32.6, 34.6).
inline int union_points(int N, int K)
{
    if (K <= 32 && N / 1000 >= K) return 4;
    return K <= 64 && N / 500 >= K ? 2 : 1;
}

// The stored neighbours of a point as a table in LDS of 2^bits slots, 8 per neighbour: of those that fall on the same slot the last one
// written is there, the others (two per row of 32) are listed.  Whether a column is among them is one read, where comparing it
// with all of them takes 104 instructions at K = 32.
constexpr int kTableMostK = 128;
inline int table_bits(int K)
{
    int bits = 4;
    while ((1 << bits) < 8 * K) ++bits;
    return bits;
}
__device__ __forceinline__ int table_slot(int c, int bits) { return (int)(((uint32_t)c * 2654435761u) >> (32 - bits)); }

// len[p] = entries of row p; len[N] = 0.  Entries of the reversed graph that add nothing to row p get bit 31 in rev.
// TABLE: PTS K at most kTableMostK; LDS of a wavefront: PTS tables, listed neighbours and the points they belong to [2 PTS K].
// Otherwise PTS = 1, and the stored neighbours are in LDS as they are.
template <int PTS, bool TABLE>
__global__ __launch_bounds__(256) void k_union_len(const int* __restrict__ idx, int N, int K, int drop_self, const int* __restrict__ offs,
                                                   int* __restrict__ rev, uint32_t div_m, int div_s, int lds_ints, int bits,
                                                   int* __restrict__ len, UnionLists L)
{
    extern __shared__ __align__(16) int union_lds[];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p0 = ((int)blockIdx.x * 4 + wave) * PTS;
    if (p0 == 0 && lane == 0) len[N] = 0;
    if (p0 >= N) return;
    int* own = union_lds + wave * lds_ints;
    int* listed = own + (PTS << bits);
    const int off = offs[min(p0 + min(lane, PTS), N)];
    int at[PTS + 1];
#pragma unroll
    for (int j = 0; j <= PTS; ++j) at[j] = read_lane_i(off, j);
    const int r0 = at[0], r1 = at[PTS];
    constexpr int kAhead = 4;
    int e[kAhead];
    auto request = [&](int r) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) e[u] = r + 64 * u + lane < r1 ? rev[r + 64 * u + lane] : -1;
    };
    request(r0);
    int n[PTS], n_listed = 0;
#pragma unroll
    for (int j = 0; j < PTS; ++j) n[j] = 0;
    if constexpr (TABLE) {
        constexpr int kOwn = kTableMostK / 64;
        int c[kOwn], mine[kOwn];
        bool ok[kOwn];
#pragma unroll
        for (int v = 0; v < kOwn; ++v) {
            const int i = lane + 64 * v;
            mine[v] = PTS == 1 ? 0 : (int)(((uint64_t)(uint32_t)i * div_m) >> div_s);       // i / K
            const bool in = i < PTS * K && p0 + mine[v] < N;
            c[v] = in ? idx[(size_t)p0 * K + i] : -1;
        }
        for (int i = 4 * lane; i < (PTS << bits); i += 256) *reinterpret_cast<int4*>(own + i) = make_int4(-1, -1, -1, -1);
#pragma unroll
        for (int v = 0; v < kOwn; ++v) {
            ok[v] = usable(c[v], p0 + mine[v], N, drop_self);
#pragma unroll
            for (int j = 0; j < PTS; ++j) n[j] += __popcll(ballot64(ok[v] && (PTS == 1 || mine[v] == j)));
        }
        wave_lds_sync();
#pragma unroll
        for (int v = 0; v < kOwn; ++v)
            if (ok[v]) own[(mine[v] << bits) + table_slot(c[v], bits)] = c[v];
        wave_lds_sync();
#pragma unroll
        for (int v = 0; v < kOwn; ++v) {
            const uint64_t lost = ballot64(ok[v] && own[((ok[v] ? mine[v] : 0) << bits) + table_slot(c[v], bits)] != c[v]);
            if (lost == 0) continue;
            if (lane_bit(lost)) {
                const int slot = n_listed + mask_prefix(lost);
                listed[2 * slot] = c[v];
                listed[2 * slot + 1] = mine[v];
            }
            n_listed += __popcll(lost);
        }
    } else {
        n[0] = own_edges(idx, N, K, p0, drop_self, own);
    }
    wave_lds_sync();
    int total[PTS];
#pragma unroll
    for (int j = 0; j < PTS; ++j) total[j] = n[j];
    for (int r = r0; r < r1; r += 64 * kAhead) {
        int now[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) now[u] = e[u];
        if (r + 64 * kAhead < r1) request(r + 64 * kAhead);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (r + 64 * u >= r1) continue;
            const int place = r + 64 * u + lane;
            int j = 0;
#pragma unroll
            for (int x = 1; x < PTS; ++x) j += place >= at[x] ? 1 : 0;
            const int c = (int)(((uint64_t)(uint32_t)now[u] * div_m) >> div_s);
            const uint64_t here = ballot64(now[u] >= 0);
            uint64_t not_new;
            if constexpr (TABLE) {
                not_new = ballot64(own[(j << bits) + table_slot(c, bits)] == c);
                for (int l = 0; l < n_listed; ++l) not_new |= ballot64(listed[2 * l] == c && (PTS == 1 || listed[2 * l + 1] == j));
            } else {
                not_new = in_own(own, n[0], c);
            }
            if (drop_self) not_new |= ballot64(c == p0 + j);
            not_new &= here;
            if (lane_bit(not_new)) rev[place] = now[u] | (int)0x80000000;
#pragma unroll
            for (int x = 0; x < PTS; ++x) total[x] += __popcll(here & ~not_new & (PTS == 1 ? ~0ull : ballot64(j == x)));
        }
    }
    // lane j: the result of point p0 + j
    int mine = total[0], seen = n[0] + at[1] - at[0];
#pragma unroll
    for (int j = 1; j < PTS; ++j)
        if (lane == j) {
            mine = total[j];
            seen = n[j] + at[j + 1] - at[j];
        }
    const int p = p0 + lane;
    if (lane >= PTS || p >= N) return;
    len[p] = mine;
    if (seen > kUnionBlock) {
        const unsigned long long was = atomicAdd(reinterpret_cast<unsigned long long*>(&L.ctr->hubs), (unsigned)mine | (1ull << 32));
        L.hubs[was >> 32] = make_int2(p, (int)(unsigned)was);
    } else if (mine > kUnionWave) {
        L.big[atomicAdd(&L.ctr->n_big, 1)] = p;
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
// (r0, r1: its reversed entries; row0, n_row: its place in the result; key, entry: kUnionWave + 4 each)
__device__ __forceinline__ void union_row(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K, int drop_self, int p,
                                          int r0, int r1, const int* __restrict__ rev, uint32_t div_m, int div_s, int row0, int n_row, int* key,
                                          int* entry, int* __restrict__ cols, float* __restrict__ vals)
{
    if (n_row == 0 || n_row > kUnionWave) return;
    const int lane = threadIdx.x & 63;
    const int e0 = r0 + lane < r1 ? rev[r0 + lane] : -1;
    int n = 0;
    for (int k0 = 0; k0 < K; k0 += 64) {
        const int k = k0 + lane;
        const int c = k < K ? idx[(size_t)p * K + k] : -1;
        const bool ok = usable(c, p, N, drop_self);
        const uint64_t m = ballot64(ok);
        if (ok) {
            const int at = n + mask_prefix(m);
            key[at] = c;
            entry[at] = p * K + k;
        }
        n += __popcll(m);
    }
    int total = n;
    for (int r = r0; r < r1; r += 64) {
        const int e = r == r0 ? e0 : (r + lane < r1 ? rev[r + lane] : -1);
        const int c = (int)(((uint64_t)(uint32_t)e * div_m) >> div_s);
        const uint64_t m = ballot64(e >= 0);                             // (k_union_len has marked those that add nothing)
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

__global__ __launch_bounds__(256) void k_union_fill(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                    int drop_self, const int* __restrict__ offs, const int* __restrict__ rev,
                                                    uint32_t div_m, int div_s, const int* __restrict__ indptr,
                                                    long long cap, int* __restrict__ cols, float* __restrict__ vals)
{
    __shared__ __align__(16) int lds[4][2 * (kUnionWave + 4)];
    if (indptr[N] > cap) return;                                        // (the host reports)
    const int wave = threadIdx.x >> 6, p = (int)blockIdx.x * 4 + wave;
    if (p >= N) return;
    const int row0 = indptr[p];
    union_row(idx, dist, N, K, drop_self, p, offs[p], offs[p + 1], rev, div_m, div_s, row0, indptr[p + 1] - row0, lds[wave],
              lds[wave] + kUnionWave + 4, cols, vals);
}

// The same for PTS points per wavefront, PTS K <= 128, whose rows have at most kUnionWave entries and kUnionFew together (others go one by
// one, as above).  LDS of a wavefront: keys and entries, each row from a multiple of four on.
constexpr int kUnionFew = 448;
template <int PTS>
__global__ __launch_bounds__(256) void k_union_fill_few(const int* __restrict__ idx, const float* __restrict__ dist, int N, int K,
                                                        int drop_self, const int* __restrict__ offs, const int* __restrict__ rev,
                                                        uint32_t div_m, int div_s, const int* __restrict__ indptr,
                                                        long long cap, int* __restrict__ cols, float* __restrict__ vals)
{
    constexpr int kRoom = kUnionFew + 4 * PTS;
    __shared__ __align__(16) int lds[4][2 * kRoom];
    if (indptr[N] > cap) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p0 = ((int)blockIdx.x * 4 + wave) * PTS;
    if (p0 >= N) return;
    int* key = lds[wave];
    int* entry = key + kRoom;
    const int off = offs[min(p0 + min(lane, PTS), N)], ind = indptr[min(p0 + min(lane, PTS), N)];
    int at[PTS + 1], row[PTS + 1], first[PTS + 1];                       // reversed entries, rows in the result, rows in LDS
    bool few = true;
    first[0] = 0;
#pragma unroll
    for (int j = 0; j <= PTS; ++j) {
        at[j] = read_lane_i(off, j);
        row[j] = read_lane_i(ind, j);
        if (j > 0) {
            first[j] = first[j - 1] + ((row[j] - row[j - 1] + 3) & ~3);
            few = few && row[j] - row[j - 1] <= kUnionWave;
        }
    }
    if (!few || row[PTS] - row[0] > kUnionFew) {
        for (int j = 0; j < PTS; ++j) {
            wave_lds_sync();
            if (p0 + j < N) union_row(idx, dist, N, K, drop_self, p0 + j, at[j], at[j + 1], rev, div_m, div_s, row[j], row[j + 1] - row[j], key, entry, cols, vals);
        }
        return;
    }
    const int r1 = at[PTS];
    constexpr int kOwn = 2, kAhead = 4;
    int c[kOwn], mine[kOwn], e[kAhead];
#pragma unroll
    for (int v = 0; v < kOwn; ++v) {
        const int i = lane + 64 * v;
        mine[v] = (int)(((uint64_t)(uint32_t)i * div_m) >> div_s);
        c[v] = i < PTS * K && p0 + mine[v] < N ? idx[(size_t)p0 * K + i] : -1;
    }
    auto request = [&](int r) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) e[u] = r + 64 * u + lane < r1 ? rev[r + 64 * u + lane] : -1;
    };
    request(at[0]);
    int next[PTS];                                                       // where the next entry of a row goes
#pragma unroll
    for (int j = 0; j < PTS; ++j) next[j] = first[j];
    auto put = [&](bool ok, int j, int col, int ent) {
        int to = 0;
#pragma unroll
        for (int x = 0; x < PTS; ++x) {
            const uint64_t m = ballot64(ok && j == x);
            to = j == x ? next[x] + mask_prefix(m) : to;
            next[x] += __popcll(m);
        }
        if (ok) {
            key[to] = col;
            entry[to] = ent;
        }
    };
#pragma unroll
    for (int v = 0; v < kOwn; ++v) put(usable(c[v], p0 + mine[v], N, drop_self), mine[v], c[v], p0 * K + lane + 64 * v);
    for (int r = at[0]; r < r1; r += 64 * kAhead) {
        int now[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) now[u] = e[u];
        if (r + 64 * kAhead < r1) request(r + 64 * kAhead);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (r + 64 * u >= r1) continue;
            const int place = r + 64 * u + lane;
            int j = 0;
#pragma unroll
            for (int x = 1; x < PTS; ++x) j += place >= at[x] ? 1 : 0;
            put(now[u] >= 0, j, (int)(((uint64_t)(uint32_t)now[u] * div_m) >> div_s), now[u]);
        }
    }
    // (what fills a row up to a multiple of four counts for nobody)
#pragma unroll
    for (int j = 0; j < PTS; ++j)
        if (lane < first[j + 1] - next[j]) key[next[j] + lane] = 0x7fffffff;
    wave_lds_sync();
    const int n = first[PTS];
    for (int i0 = 0; i0 < n; i0 += 128) {
        int k[2], rank[2], to[2], s0[2], s1[2];
        float v[2];
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int i = i0 + 64 * x + lane;
            k[x] = i < n ? key[i] : 0x7fffffff;
            v[x] = k[x] != 0x7fffffff && dist ? dist[entry[i]] : 0.0f;
            rank[x] = 0;
            to[x] = row[0];
            s0[x] = 0;
            s1[x] = first[1];
#pragma unroll
            for (int y = 1; y < PTS; ++y)
                if (i >= first[y]) {
                    to[x] = row[y];
                    s0[x] = first[y];
                    s1[x] = first[y + 1];
                }
            if (k[x] == 0x7fffffff) s1[x] = s0[x];
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
            for (int j = s0[x]; j < s1[x]; j += 4) {
                const int4 o = *reinterpret_cast<const int4*>(key + j);
                rank[x] += o.x < k[x] ? 1 : 0;
                rank[x] += o.y < k[x] ? 1 : 0;
                rank[x] += o.z < k[x] ? 1 : 0;
                rank[x] += o.w < k[x] ? 1 : 0;
            }
#pragma unroll
        for (int x = 0; x < 2; ++x)
            if (k[x] != 0x7fffffff) {
                cols[to[x] + rank[x]] = k[x];
                vals[to[x] + rank[x]] = v[x];
            }
    }
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
            if (e >= 0) a[atomicAdd(&n_s, 1)] = ((unsigned long long)(unsigned)c << 32) | 0x80000000ull | (unsigned)e;
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
                                                    uint32_t div_m, int div_s, const int2* __restrict__ hubs, int col_bits,
                                                    int* __restrict__ cursor, unsigned long long* __restrict__ keys,
                                                    float* __restrict__ vals)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.x, p = hubs[h].x, first = hubs[h].y;
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
        put(e >= 0, c, e);
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
    int* rev = explore_ws_rev(rg.w);
    // e / K for 0 <= e < 2^30
    int l = 0;
    while ((1 << l) < K) ++l;
    const int div_s = 31 + l;
    const uint32_t div_m = (uint32_t)((((uint64_t)1 << div_s) + (uint64_t)K - 1) / (uint64_t)K);
    const int pts = union_points(N, K), bits = table_bits(K);
    const unsigned grid = (unsigned)((N + 4 * pts - 1) / (4 * pts));
    const int len_ints = K <= kTableMostK ? (pts << bits) + ((2 * pts * K + 3) & ~3) : (K + 4 + 3) & ~3;
#define RSFK_UNION_LEN(PTS, TABLE)                                                                                          \
    hipLaunchKernelGGL((k_union_len<PTS, TABLE>), dim3(grid), dim3(256), (size_t)4 * len_ints * sizeof(int), stream, d_idx, N, K,  \
                       drop_self, offs, rev, div_m, div_s, len_ints, TABLE ? bits : 0, static_cast<int*>(len.p), L)
    if (pts == 4) RSFK_UNION_LEN(4, true);
    else if (pts == 2) RSFK_UNION_LEN(2, true);
    else if (K <= kTableMostK) RSFK_UNION_LEN(1, true);
    else RSFK_UNION_LEN(1, false);
#undef RSFK_UNION_LEN
    RSFK_HIP(hipGetLastError());
    size_t tmp_bytes = 0;
    RSFK_HIP(rocprim::exclusive_scan(nullptr, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                     rocprim::plus<int>(), stream));
    Buf tmp;
    if (ws_alloc(&tmp.p, tmp_bytes ? tmp_bytes : 256)) return 1;
    RSFK_HIP(rocprim::exclusive_scan(tmp.p, tmp_bytes, static_cast<int*>(len.p), d_indptr, 0, (size_t)N + 1,
                                     rocprim::plus<int>(), stream));
    const auto fill = [&]() -> int {
        if (pts == 4)
            hipLaunchKernelGGL(k_union_fill_few<4>, dim3(grid), dim3(256), 0, stream, d_idx, d_dist, N, K, drop_self, offs, rev, div_m, div_s,
                               d_indptr, out.cap, out.cols, out.vals);
        else if (pts == 2)
            hipLaunchKernelGGL(k_union_fill_few<2>, dim3(grid), dim3(256), 0, stream, d_idx, d_dist, N, K, drop_self, offs, rev, div_m, div_s,
                               d_indptr, out.cap, out.cols, out.vals);
        else
            hipLaunchKernelGGL(k_union_fill, dim3(grid), dim3(256), 0, stream, d_idx, d_dist, N, K, drop_self, offs, rev, div_m, div_s,
                               d_indptr, out.cap, out.cols, out.vals);
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
        hipLaunchKernelGGL(k_hub_gather, dim3((unsigned)n_hubs, shares), dim3(256), 0, stream, d_idx, d_dist,
                           N, K, drop_self, offs, rev, div_m, div_s, L.hubs, col_bits, static_cast<int*>(cursor.p), key[0], val[0]);
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
    // (the sort has a workgroup for a row: rows in pieces that a launch has threads for)
    constexpr int kSortRows = 1 << 22;
    size_t sort_bytes = 0;
    RSFK_HIP(rocprim::segmented_radix_sort_pairs(nullptr, sort_bytes, static_cast<int*>(cols.p), d_cols,
                                                 static_cast<float*>(vals.p), d_vals, (unsigned)n, (unsigned)std::min(N, kSortRows), d_indptr,
                                                 d_indptr + 1, 0, (unsigned)bits, stream));
    Buf tmp;
    if (ws_alloc(&tmp.p, sort_bytes ? sort_bytes : 256)) return 1;
    for (int first = 0; first < N; first += std::min(kSortRows, N - first))
        RSFK_HIP(rocprim::segmented_radix_sort_pairs(tmp.p, sort_bytes, static_cast<int*>(cols.p), d_cols,
                                                     static_cast<float*>(vals.p), d_vals, (unsigned)n, (unsigned)std::min(kSortRows, N - first),
                                                     d_indptr + first, d_indptr + first + 1, 0, (unsigned)bits, stream));
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
