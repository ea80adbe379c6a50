// Candidate generation for the neighbourhood exploration as a join over the reversed
// graph.  Same candidates as nearest_neighbors_exploring
// (src/kernels/nearest_neighbors_exploring.cu:41-146) looks at -- for a point p the
// neighbours c of its neighbours q -- but enumerated from the middle: for every q, all
// pairs (p, c) with p in R(q) = {points that list q} and c in N(q).  The rows of N(q)
// and R(q) are then loaded once per q instead of once per pair, and the pair distances
// of a 32 x 32 tile come from one chain of matrix-core instructions on the float16
// copy of the points (v_mfma_f32_32x32x16_f16: Gram matrix G, d~ = n_p + n_c - 2 G).
//
// d~ is only used to discard.  All in the units of the copy (join_copy.hpp: distances times s^2), with S = n_p + n_c (norms of its
// rows) and e_p, e_c what rounding took from the two rows:
//   rounding to float16:    sqrt(d(real)) >= sqrt(d~(real)) - e_p - e_c  (triangle inequality)
//   Gram matrix and norms:  |d~(computed) - d~(real)| <= E1 = (D' + 16) 2^-21 S
//   fp32 chain:             result >= d(real) (1 - gamma),  gamma = (D + 8) 2^-22
// so a pair is dropped when d~ - E1 is above (bar_p + e_c)^2, bar_p = s sqrt(last slot of row p / (1 - gamma)) + e_p: its exact
// distance is then above the last slot.  For e the smaller is taken of what holds for any row of that norm, 2^-11 |row| + 2^-14 sqrt(D),
// and of the largest length measured when the copy was made; norms come from the rows themselves, which the kernels have in registers.
// So the bar, four bytes, is all that is gathered besides the rows.  (Records of norm and bar for both sides: 1M x 256
// 8.0 -> 7.0 ms, 10M x 32 27.2 -> 24.6, 1M x 100 3.66 -> 3.45.)
// (Measured against rows in bfloat16 with 2^-8 |row| for e: exact distances per point 1M x 100 28 -> 22, 1M x 256 in 64 clusters
// 74 -> 39, sparse 70,000 x 784 with K = 90 185 -> 140, 10M x 32 49 -> 42; merge 3.54 -> 2.77, 13.9 -> 8.25, 15.9 -> 12.6 and 23.6 ->
// 20.1 ms.  bfloat16 with the measured e: 24, 41, 147 and 45.)
// The outcome is one bit per (entry of the graph, neighbour slot): pass[p K + k] for the
// entry (p, k) = q has bit n set iff neighbour n of q may enter row p (an element of R(q)
// is the number p K + k of the entry, so the join knows where to write and the merge
// kernel of p reads its K words in one piece).  The exploration kernel of point p gathers
// the few ids whose bit is set (a few per cent), computes their exact distances and
// merges them.  Nothing is decided here that the exact arithmetic would decide
// otherwise; no atomics on shared counters, no buffer that can overflow.
//
// What the row certainly holds is not marked: q itself (in its own row as a rule, and in row p for every p in R(q)), and everything where p is q.
// That is half of what passes the bound or more, and in every word: each such mark was an id gathered by the merge, and the words that are
// left without marks are not stored (k_join_bars clears them).  (Their norms are taken for kNever, so a row with an infinite bar keeps such marks, and the
// merge drops them.)  p among the neighbours of q, which the merge would drop too, is found by JoinSelf.
// 10M x 32: join 24.7 -> 23.1 ms, merge 20.3 -> 18.9; 1M x 100 3.39 -> 3.21, 2.76 -> 2.56; 1M x 256 7.14 -> 7.05, 6.04 -> 5.93; 20,000 x 32 merge 0.086 -> 0.046;
// 70,000 x 784, K = 90 the same.  (A fifth of the words is left without marks at 10M x 32: most others hold points that row p has from elsewhere.)
//
// For the merge kernel that works through a point's candidates in the order of their
// bounds (explore.hip: rows with many candidates), the bound is kept for every marked
// pair as a 16-bit code (join_bounds.hpp).
//
// Steps: R in compressed rows (counting sort of the graph entries by neighbour, see k_bin_count) -> join.
#include "rsfk_common.hpp"
#include "wave64.hpp"
#include "forest.hpp"
#include "join_bounds.hpp"
#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace rsfk {

struct ExploreWorkspace {
    int N = 0, K = 0, MW = 0;  // MW = 32-bit words per entry of pass
    int shift = 0;             // a bin of the reversed-graph builder = 2^shift consecutive points
    int n_bins = 0;
    int n_parts = 0;           // workgroups of the two passes over the graph; each owns a contiguous range of entries
    int per_part = 0;          // entries per such range
    uint32_t div_m = 0;        // e / K == (div_m * e) >> div_s for 0 <= e < 2^31
    int div_s = 0;
    int* rev = nullptr;        // N*K: R lists in compressed rows; an element is the number p K + k of a graph entry
    uint16_t* rev_bars = nullptr;   // N*K: code of the bar of the point of each element of rev (bar_code), or null
    int* offs = nullptr;       // N+1: start of R(q)
    int2* bin_eq = nullptr;    // N*K: (entry number, neighbour minus the first point of its bin), grouped by the bin of
                               // the neighbour; one 8-byte store per entry
    int* bin_size = nullptr;   // n_bins
    int* bin_start = nullptr;  // n_bins + 1
    int* part_off = nullptr;   // n_parts x n_bins: where the entries of a part start inside a bin
    uint32_t* pass = nullptr;  // N*K*MW, indexed by entry number
    float* bars = nullptr;     // N: the bar the candidates of a point have to pass (k_join_bars)
    JoinBounds view;           // what the merge kernels read (set by launch_explore_join)
    uint16_t* bounds = nullptr; // N*K*32*MW codes of the marked pairs (join_bounds.hpp), or null
    int direct = 0;             // the builder of small graphs: points of a workgroup, or 0
    bool tiled = false;         // the builder of medium graphs: bins of 2^cshift points, rows of 2^fshift of them at a time
    // the builder for large graphs (staged_rev_*): two scatters through LDS instead of one straight to memory
    bool staged = false;
    int fshift = 0, cshift = 0; // fine bins of 2^fshift points (their rows are assembled in LDS), coarse bins of 2^cshift
    int n_fine = 0, n_coarse = 0;
    int n_sub = 0;              // sub-parts of the coarse bins at the second level (an upper bound)
    int2* bin_eq2 = nullptr;    // N*K: the records grouped by fine bin
    int* fine_size = nullptr;   // n_coarse << (cshift - fshift)
    int* fine_start = nullptr;  // the same + 1
    int* sub_off = nullptr;     // n_sub x fine bins per coarse bin
    int* todo = nullptr;       // two lists of N + 1 ints, points left over by a launch (entry N of the second: their number); then the
                               // shares from which the first is joined, and their numbers
};
int* explore_ws_shares(ExploreWorkspace* w)
{
    const size_t at = 2 * ((size_t)w->N + 1) + (size_t)kTodoShares * (size_t)todo_share(w->N);
    return w->todo + ((at + 31) & ~(size_t)31);
}
namespace {

size_t todo_ints(int N) { return 2 * ((size_t)N + 1) + (size_t)kTodoShares * (size_t)todo_share(N) + 32 + 32 * (size_t)kTodoShares; }

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

constexpr int kMaxBins = 6144;
constexpr int kMaxShift = 13;
// entry numbers are ints, and the passes over the graph look up to 4,095 entries beyond the one they test (the staged scatters and rows; k_bin_count 3,072)
constexpr size_t kMaxEntries = ((size_t)1 << 31) - 4096;
// entries of the largest graph that k_rev_direct takes
constexpr size_t kDirectMost = (size_t)1 << 18;
constexpr int kRowsBlock = 512;             // threads of k_bin_rows

// RSFK_JOIN_WG=0: the wavefront-per-q join also where the workgroup-per-q one applies.
bool join_wg_on()
{
    static const bool on = [] {
        const char* e = std::getenv("RSFK_JOIN_WG");
        return !(e && e[0] == '0');
    }();
    return on;
}

// Bins of the reversed-graph builder for N points: false if N is too large for it.
bool rev_bins(int N, int* shift, int* n_bins)
{
    // measured: small bins make the placement of k_bin_rows local (1M points: 0.25 ms with bins of 256 points, 0.62 ms
    // with 1024), many bins make the runs k_bin_scatter writes short (0.49 against 0.36 ms)
    int s = 8;
    if (const char* e = std::getenv("RSFK_REV_SHIFT")) s = std::max(8, std::min(kMaxShift, std::atoi(e)));
    while (s < kMaxShift && (((N - 1) >> s) + 1) > kMaxBins) ++s;
    *shift = s;
    *n_bins = N > 0 ? ((N - 1) >> s) + 1 : 1;
    return *n_bins <= kMaxBins;
}

// A bar in 16 bits, rounded up: 11 bits behind the leading one, from 2^-9 to 2^23 (in the units of the copy, whose coordinates are below 2^15 and
// not all below 2^12); what is not below that, or NaN, is infinite.  A candidate more passes for it, none less.  (10M x 32: 0.8 % more marks.)
// The staged builder of the reversed graph carries it beside the entries, in the half of a record that the place in its bin leaves, because it
// reads the graph point by point: gathered by the join, the bars are a line read for every element of R(q), and a trip after it.
// 10M x 32: join 15.54 -> 12.02 ms, last step of the builder 2.24 -> 2.54.  (Smaller graphs, whose bars stay in the L2, gain nothing: 1M x 100 join 2.86 ->
// 2.85 ms, last step of the builder 0.18 -> 0.25.)
constexpr uint32_t kBarBase = 118u << 11;
__device__ __forceinline__ uint32_t bar_code(float bar)
{
    if (!(bar < 8388608.0f)) return 0xffffu;
    return min(((__float_as_uint(fmaxf(bar, 1.0f / 512.0f)) + 0xfffu) >> 12) - kBarBase, 0xffffu);
}
__device__ __forceinline__ float bar_of(uint32_t code) { return code == 0xffffu ? INFINITY : __uint_as_float((code + kBarBase) << 12); }

// What a builder needs for it.  With bars a record's second word is the place in its bin (16 bits) and the code above it.
struct RevBars {
    const float* bars = nullptr;
    uint32_t div_m = 0;
    int div_s = 0;
    __device__ __forceinline__ float of_entry(int e) const { return bars[(int)(((uint64_t)div_m * (uint64_t)(uint32_t)e) >> div_s)]; }
};

__global__ void k_zero(int* a, int n, int* counter, int* shares)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
    if (i == 0) *counter = 0;
    if (i < kTodoShares) shares[32 * i] = 0;
}

// exclusive scan of one value per thread over the workgroup (blockDim.x a multiple of 64, at most 1024); returns the
// total in *total.  lds: one int per wavefront.
__device__ __forceinline__ int block_excl_scan(int v, int* total, int* lds)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    int incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) lds[wave] = incl;
    __syncthreads();
    int woff = 0, tot = 0;
    for (int w = 0; w < waves; ++w) { const int x = lds[w]; if (w < wave) woff += x; tot += x; }
    __syncthreads();
    *total = tot;
    return woff + incl - v;
}

// The reversed graph R(q) = {entries (p, k) of the graph that hold q}, in compressed rows, without an atomic operation
// on device memory per entry (device-wide atomics are carried out at the memory side of the fabric, about 27 G of them
// a second: 2.8 ms for the 32 M entries of a 1 M x 32 graph, counting and placing).  Counting sort in two levels:
// the points are cut into bins of 2^shift, (1) every part of the graph counts its entries per bin in LDS and reserves
// its share of each bin with one atomic per bin, (2) the entries are moved to their bins -- entry number and neighbour
// minus the start of the bin -- (3) one workgroup per bin counts its neighbours in LDS, scans, writes the row offsets
// and places the entries.  The order of the entries inside R(q) is arbitrary; nothing downstream depends on it.
__global__ __launch_bounds__(1024) void k_bin_count(const int* __restrict__ old_idx, int total, int per_part, int N, int shift,
                                                   int n_bins, int* __restrict__ bin_size, int* __restrict__ part_off)
{
    extern __shared__ int hist[];
    for (int b = threadIdx.x; b < n_bins; b += blockDim.x) hist[b] = 0;
    __syncthreads();
    const long long first = (long long)blockIdx.x * per_part;
    const int e0 = (int)min((long long)total, first), e1 = (int)min((long long)total, first + per_part);
    for (int e = e0 + (int)threadIdx.x; e < e1; e += 4 * (int)blockDim.x) {
        int q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = e + (int)blockDim.x * u < e1 ? old_idx[e + (int)blockDim.x * u] : -1;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (q[u] >= 0 && q[u] < N) atomicAdd(&hist[q[u] >> shift], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < n_bins; b += blockDim.x) {
        const int c = hist[b];
        part_off[(size_t)blockIdx.x * n_bins + b] = c ? atomicAdd(&bin_size[b], c) : 0;
    }
}

// bin_start = exclusive scan of bin_size (one workgroup); the number of valid entries goes to bin_start[n_bins] and *last
__global__ __launch_bounds__(256) void k_bin_scan(const int* __restrict__ bin_size, int n_bins, int* __restrict__ bin_start,
                                                  int* __restrict__ last)
{
    __shared__ int lds4[4];
    int carry = 0;
    for (int b0 = 0; b0 < n_bins; b0 += 256) {
        const int i = b0 + threadIdx.x;
        const int v = i < n_bins ? bin_size[i] : 0;
        int tot;
        const int ex = block_excl_scan(v, &tot, lds4);
        if (i < n_bins) bin_start[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) { bin_start[n_bins] = carry; *last = carry; }
}

__global__ __launch_bounds__(256) void k_bin_scatter(const int* __restrict__ old_idx, int total, int per_part, int N, int shift,
                                                     int n_bins, const int* __restrict__ bin_start,
                                                     const int* __restrict__ part_off, int2* __restrict__ bin_eq)
{
    extern __shared__ int cursor[];
    for (int b = threadIdx.x; b < n_bins; b += 256) cursor[b] = bin_start[b] + part_off[(size_t)blockIdx.x * n_bins + b];
    __syncthreads();
    const int low = (1 << shift) - 1;
    const long long first = (long long)blockIdx.x * per_part;
    const int e0 = (int)min((long long)total, first), e1 = (int)min((long long)total, first + per_part);
    for (int e = e0 + (int)threadIdx.x; e < e1; e += 1024) {
        int q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = e + 256 * u < e1 ? old_idx[e + 256 * u] : -1;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (q[u] >= 0 && q[u] < N) {
                const int at = atomicAdd(&cursor[q[u] >> shift], 1);
                bin_eq[at] = make_int2(e + 256 * u, q[u] & low);
            }
        }
    }
}

// One workgroup per bin.  LDS: one counter per point of the bin.
__global__ __launch_bounds__(kRowsBlock) void k_bin_rows(const int2* __restrict__ bin_eq,
                                                         const int* __restrict__ bin_start, int shift, int N,
                                                         int* __restrict__ offs, int* __restrict__ rev)
{
    extern __shared__ int cnt[];
    __shared__ int wave_lds[kRowsBlock / 64];
    const int R = 1 << shift;
    const int b = blockIdx.x;
    const int s0 = bin_start[b], s1 = bin_start[b + 1];
    const int q0 = b << shift;
    for (int i = threadIdx.x; i < R; i += kRowsBlock) cnt[i] = 0;
    __syncthreads();
    for (int i = s0 + (int)threadIdx.x; i < s1; i += kRowsBlock) atomicAdd(&cnt[bin_eq[i].y], 1);
    __syncthreads();
    int carry = 0;
    for (int c0 = 0; c0 < R; c0 += kRowsBlock) {
        const int c = c0 + (int)threadIdx.x;
        const bool in = c < R;                            // (a bin may have fewer points than the workgroup has threads)
        const int v = in ? cnt[c] : 0;
        int tot;
        const int ex = block_excl_scan(v, &tot, wave_lds);
        if (in) {
            cnt[c] = carry + ex;
            if (q0 + c < N) offs[q0 + c] = s0 + carry + ex;
        }
        carry += tot;
    }
    __syncthreads();
    for (int i = s0 + (int)threadIdx.x; i < s1; i += kRowsBlock) {
        const int2 eq = bin_eq[i];
        const int at = atomicAdd(&cnt[eq.y], 1);
        rev[s0 + at] = eq.x;
    }
}

// ---------------------------------------------------------------------------
// The same reversed graph for small inputs, in one launch.  What bounds the five above there is their launches.  A workgroup has `per` points and goes
// through the whole graph (from the L2): it counts the entries of the points before its own, which is where its rows begin, and lists the numbers of its
// own in LDS, which are then counted, scanned and placed; if they are more than fit, it goes through the graph twice more.
// Points x neighbours, us in one launch and the kernels of the five: 3,000 x 30 13 and 29, 10,000 x 16 17 and 25, 8,000 x 25 21 and 28, 16,000 x 16 (256,000 entries) 24.9 and
// 25.4, 2,600 x 100 25 and 51, 8,200 x 32 25 and 31, 20,000 x 16 (320,000) 30 and 26, 10,000 x 32 29 and 31, 40,000 x 10 36 and 26, 14,000 x 32 39 and 29, 20,000 x 32 (640,000) 53 and
// 33: up to 2^18 entries.  (Bound by its instructions, six per entry in every workgroup: a branch and an addition per entry instead 15, 21 and 60 us for 3,000 x 30,
// 10,000 x 16 and 20,000 x 32; the next entries on their way, or workgroups that begin in different places, the same.)
constexpr int kDirectThreads = 1024, kDirectCap = 8192, kDirectMostPer = 4096;
typedef int i32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

__global__ __launch_bounds__(kDirectThreads) void k_rev_direct(const int* __restrict__ old_idx, int total, int N, int per, int* __restrict__ offs,
                                                               int* __restrict__ rev, int* counter, int* shares)
{
    extern __shared__ int cnt[];                          // entries of each point, then where its next one goes
    __shared__ int own[kDirectCap];
    __shared__ int wave_lds[kDirectThreads / 64];
    __shared__ int n_own;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lo = blockIdx.x * per, n = min(N - lo, per);
    if (blockIdx.x == 0) {
        if (tid == 0) *counter = 0;
        if (tid < kTodoShares) shares[32 * tid] = 0;
    }
    for (int i = tid; i < n; i += kDirectThreads) cnt[i] = 0;
    if (tid == 0) n_own = 0;
    __syncthreads();
    int below = 0;
    for (int t0 = 4 * tid; t0 < total; t0 += 16 * kDirectThreads) {
        i32x4_a4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int e = t0 + 4 * kDirectThreads * u;
            if (e + 4 <= total) {
                q[u] = *reinterpret_cast<const i32x4_a4*>(old_idx + e);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) q[u][j] = e + j < total ? old_idx[e + j] : -1;
            }
        }
        // (no branch per entry: one in `per` of N is this workgroup's, a few of the thousand of a wavefront)
        uint32_t hits = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int c = q[i >> 2][i & 3];
            below += (unsigned)c < (unsigned)lo ? 1 : 0;
            hits |= (unsigned)(c - lo) < (unsigned)n ? 1u << i : 0u;
        }
        while (hits) {
            const int i = __builtin_ctz(hits);
            hits &= hits - 1;
            const int at = atomicAdd(&n_own, 1);
            if (at < kDirectCap) own[at] = t0 + 4 * kDirectThreads * (i >> 2) + (i & 3);
        }
    }
    below = wave_sum_i(below);
    if (lane == 0) wave_lds[wave] = below;
    __syncthreads();
    int begin = 0;
    for (int w = 0; w < kDirectThreads / 64; ++w) begin += wave_lds[w];
    const int m = n_own;
    // calls f(entry, place of its point) for the workgroup's entries
    const auto for_own = [&](auto f) {
        if (m <= kDirectCap) {
            for (int i = tid; i < m; i += kDirectThreads) f(own[i], old_idx[own[i]] - lo);
        } else {
            for (int e = tid; e < total; e += kDirectThreads) {
                const int c = old_idx[e] - lo;
                if ((unsigned)c < (unsigned)n) f(e, c);
            }
        }
    };
    for_own([&](int, int c) { atomicAdd(&cnt[c], 1); });
    __syncthreads();
    int carry = begin;
    for (int c0 = 0; c0 < n; c0 += kDirectThreads) {
        const int c = c0 + tid, v = c < n ? cnt[c] : 0;
        int all;
        const int ex = block_excl_scan(v, &all, wave_lds);
        if (c < n) {
            cnt[c] = carry + ex;
            offs[lo + c] = carry + ex;
        }
        carry += all;
    }
    if (lo + n == N && tid == 0) offs[N] = carry;
    __syncthreads();
    for_own([&](int e, int c) { rev[atomicAdd(&cnt[c], 1)] = e; });
}

// ---------------------------------------------------------------------------
// The same reversed graph for large inputs.  k_bin_scatter sends every record straight to one of several thousand
// bins and k_bin_rows every entry straight to its row: stores of 8 and 4 bytes whose cache lines leave the L2 long
// before their neighbours arrive (10 M x 32: 9.4 GB and 8.6 GB written for 2.56 GB and 1.28 GB of payload).  Here
// every store to memory is a run: (1) the records go to a few hundred coarse bins, a tile of 4096 at a time sorted by
// bin in LDS first, so a bin receives a run of records per tile; (2) inside a coarse bin the same again to its fine
// bins; (3) a fine bin is small enough for all of its rows to be assembled in LDS and written whole.  Counting comes
// before every scatter as in the one-level builder (no atomics on device memory per entry).  A record is
// (entry number, neighbour).
constexpr int kStTile = 4096;               // records sorted in LDS at a time
constexpr int kStSub = 32768;               // records of a sub-part of a coarse bin
constexpr int kStMaxBins = 1024;            // bins a scatter step distinguishes (LDS counters)
constexpr int kStRowsCap = 24576;           // entries of a fine bin whose rows are assembled in LDS

// (The counts of the parts of the graph per coarse bin are k_bin_count and k_bin_scan with shift = cshift.)

// Sorts up to kStTile records (rec[i], bin[i] for the thread's 16 records) by bin in LDS and writes them to
// out[cursor[bin] + rank inside (tile, bin)]; cursor (LDS, n_bins ints) moves on by the tile's counts.
// LDS: cnt[n_bins] | first[n_bins] | stage[kStTile] (int2).
__device__ __forceinline__ void staged_tile_out(const int2 (&rec)[16], const int (&bin)[16], int n_bins, int* cnt, int* first,
                                                int2* stage, unsigned short* sbin, int* cursor, int* wave_lds,
                                                int2* __restrict__ out)
{
    const int tid = threadIdx.x;
    for (int b = tid; b < n_bins; b += 256) cnt[b] = 0;
    __syncthreads();
    int rank[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) rank[u] = bin[u] >= 0 ? atomicAdd(&cnt[bin[u]], 1) : 0;
    __syncthreads();
    // exclusive scan of the counts (n_bins <= 1024: four per thread)
    {
        int v[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) { const int b = 4 * tid + j; v[j] = b < n_bins ? cnt[b] : 0; sum += v[j]; }
        int tot;
        int ex = block_excl_scan(sum, &tot, wave_lds);
#pragma unroll
        for (int j = 0; j < 4; ++j) { const int b = 4 * tid + j; if (b < n_bins) first[b] = ex; ex += v[j]; }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        if (bin[u] >= 0) {
            const int at = first[bin[u]] + rank[u];
            stage[at] = rec[u];
            sbin[at] = (unsigned short)bin[u];
        }
    }
    __syncthreads();
    const int n_tile = first[n_bins - 1] + cnt[n_bins - 1];
    for (int i = tid; i < n_tile; i += 256) {
        const int b = sbin[i];
        out[(size_t)cursor[b] + (size_t)(i - first[b])] = stage[i];
    }
    __syncthreads();
    for (int b = tid; b < n_bins; b += 256) cursor[b] += cnt[b];
    __syncthreads();
}

constexpr size_t staged_lds_bytes(int n_bins)
{
    return (size_t)3 * n_bins * sizeof(int) + 8 + (size_t)kStTile * (sizeof(int2) + sizeof(unsigned short));
}

// (1) a part of the graph to the coarse bins.  part_off / bin_start as left by k_bin_count / k_bin_scan at shift = cshift.
template <bool BARS>
__global__ __launch_bounds__(256) void k_staged_scatter1(const int* __restrict__ old_idx, int total, int per_part, int N, int cshift,
                                                         int n_coarse, const int* __restrict__ bin_start,
                                                         const int* __restrict__ part_off, int2* __restrict__ out, RevBars rb)
{
    extern __shared__ __align__(16) int lds_st[];
    __shared__ int wave_lds[4];
    int* cursor = lds_st;
    int* cnt = cursor + n_coarse;
    int* first = cnt + n_coarse;
    int2* stage = reinterpret_cast<int2*>(first + n_coarse + (n_coarse & 1));
    unsigned short* sbin = reinterpret_cast<unsigned short*>(stage + kStTile);
    for (int b = threadIdx.x; b < n_coarse; b += 256) cursor[b] = bin_start[b] + part_off[(size_t)blockIdx.x * n_coarse + b];
    __syncthreads();
    const long long begin = (long long)blockIdx.x * per_part;
    const int e0 = (int)min((long long)total, begin), e1 = (int)min((long long)total, begin + per_part);
    // (the neighbours of the next tile travel while this one is sorted)
    int q[16];
    float bar[16];
    auto request = [&](int t0) {
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int e = t0 + 256 * u + (int)threadIdx.x;
            q[u] = e < e1 ? old_idx[e] : -1;
            if (BARS) bar[u] = rb.of_entry(min(e, e1 - 1));
        }
    };
    if (e0 < e1) request(e0);
    for (int t0 = e0; t0 < e1; t0 += kStTile) {
        int2 rec[16];
        int bin[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const bool ok = q[u] >= 0 && q[u] < N;
            rec[u] = make_int2(t0 + 256 * u + (int)threadIdx.x,
                               BARS ? (int)(((uint32_t)q[u] & ((1u << cshift) - 1u)) | bar_code(bar[u]) << 16) : q[u]);
            bin[u] = ok ? q[u] >> cshift : -1;
        }
        if (t0 + kStTile < e1) request(t0 + kStTile);
        staged_tile_out(rec, bin, n_coarse, cnt, first, stage, sbin, cursor, wave_lds, out);
    }
}

// Sub-parts of coarse bin cb: records [start + s kStSub, ...) for s = 0, 1, ...; their number in the global list of
// sub-parts is start / kStSub + cb + s (increasing, no two alike: a coarse bin has at most size / kStSub + 1 of them).
__device__ __forceinline__ int staged_sub_id(int start, int cb, int s) { return start / kStSub + cb + s; }

// (2a) counts of the sub-parts of the coarse bins per fine bin; grid (x: sub-parts walked in turn, y: coarse bin)
__global__ __launch_bounds__(256) void k_staged_count2(const int2* __restrict__ rec1, const int* __restrict__ cstart, int cshift,
                                                       int fshift, int* __restrict__ fine_size, int* __restrict__ sub_off)
{
    extern __shared__ int hist2[];
    const int per = 1 << (cshift - fshift);
    const int cb = blockIdx.y;
    const int s0 = cstart[cb], s1 = cstart[cb + 1];
    const int low = (1 << cshift) - 1;
    for (int s = blockIdx.x; s0 + (long long)s * kStSub < s1; s += gridDim.x) {
        for (int b = threadIdx.x; b < per; b += 256) hist2[b] = 0;
        __syncthreads();
        const int a = s0 + s * kStSub, z = a + min(s1 - a, kStSub);
        for (int i = a + (int)threadIdx.x; i < z; i += 256) atomicAdd(&hist2[(rec1[i].y & low) >> fshift], 1);
        __syncthreads();
        const size_t row = (size_t)staged_sub_id(s0, cb, s) * per;
        for (int b = threadIdx.x; b < per; b += 256) {
            const int c = hist2[b];
            sub_off[row + b] = c ? atomicAdd(&fine_size[(size_t)cb * per + b], c) : 0;
        }
        __syncthreads();
    }
}

// (2b) the records of the sub-parts to their fine bins.  A tile of 8192 records in LDS, two workgroups per compute unit, the next tile on its way: 10M x 32
// 1.95 -> 1.29 ms against tiles of 4096 and three workgroups of half the threads.
constexpr int kSt2Threads = 512, kSt2Per = 16, kSt2Tile = kSt2Threads * kSt2Per;
__host__ __device__ inline size_t staged2_lds_bytes(int per) { return (size_t)3 * ((per + 3) & ~3) * sizeof(int) + (size_t)kSt2Tile * sizeof(int2); }

__global__ __launch_bounds__(kSt2Threads) void k_staged_scatter2(const int2* __restrict__ rec1, const int* __restrict__ cstart, int cshift,
                                                                 int fshift, const int* __restrict__ fine_start,
                                                                 const int* __restrict__ sub_off, int2* __restrict__ out)
{
    extern __shared__ __align__(16) int lds_st[];
    __shared__ int wave_lds[kSt2Threads / 64];
    const int per = 1 << (cshift - fshift), pitch = (per + 3) & ~3, tid = threadIdx.x;       // (at most 1024 fine bins: two per thread)
    int* cursor = lds_st;
    int* cnt = cursor + pitch;
    int* first = cnt + pitch;
    int2* stage = reinterpret_cast<int2*>(first + pitch);
    const int cb = blockIdx.y;
    const int s0 = cstart[cb], s1 = cstart[cb + 1];
    const int low = (1 << cshift) - 1;
    for (int s = blockIdx.x; s0 + (long long)s * kStSub < s1; s += gridDim.x) {
        const size_t row = (size_t)staged_sub_id(s0, cb, s) * per;
        for (int b = tid; b < per; b += kSt2Threads) cursor[b] = fine_start[(size_t)cb * per + b] + sub_off[row + b];
        const int a = s0 + s * kStSub, n = min(s1 - a, kStSub);
        int2 r[kSt2Per];
        auto request = [&](int t0) {
#pragma unroll
            for (int u = 0; u < kSt2Per; ++u) {
                const int i = t0 + kSt2Threads * u + tid;
                r[u] = i < n ? rec1[(size_t)a + (size_t)i] : make_int2(-1, 0);
            }
        };
        request(0);
        for (int t0 = 0; t0 < n; t0 += kSt2Tile) {
            for (int b = tid; b < per; b += kSt2Threads) cnt[b] = 0;
            __syncthreads();
            int rank[kSt2Per];
#pragma unroll
            for (int u = 0; u < kSt2Per; ++u) rank[u] = r[u].x >= 0 ? atomicAdd(&cnt[(r[u].y & low) >> fshift], 1) : 0;
            __syncthreads();
            const int b0 = 2 * tid, c0 = b0 < per ? cnt[b0] : 0, c1 = b0 + 1 < per ? cnt[b0 + 1] : 0;
            int n_tile;
            const int ex = block_excl_scan(c0 + c1, &n_tile, wave_lds);
            if (b0 < per) first[b0] = ex;
            if (b0 + 1 < per) first[b0 + 1] = ex + c0;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < kSt2Per; ++u)
                if (r[u].x >= 0) stage[first[(r[u].y & low) >> fshift] + rank[u]] = r[u];
            __syncthreads();
            if (t0 + kSt2Tile < n) request(t0 + kSt2Tile);
            for (int i = tid; i < n_tile; i += kSt2Threads) {
                const int2 x = stage[i];
                const int b = (x.y & low) >> fshift;
                out[(size_t)cursor[b] + (size_t)(i - first[b])] = x;
            }
            __syncthreads();
            for (int b = tid; b < per; b += kSt2Threads) cursor[b] += cnt[b];
            __syncthreads();
        }
    }
}

// (3) one workgroup per fine bin: row offsets of its points, and its rows -- assembled in LDS and written whole when the
// bin has at most kStRowsCap entries, entry by entry otherwise.  LDS: cnt[2^fshift] | stage[kStRowsCap] | codes[kStRowsCap] (16 bits; with bars), which leaves one
// workgroup to a compute unit: 1024 threads with four loads each in flight (10M x 32 2.54 -> 1.12 ms against 512 with one).
constexpr int kStRowsThreads = 1024;
template <bool BARS>
__global__ __launch_bounds__(kStRowsThreads) void k_staged_rows(const int2* __restrict__ rec2, const int* __restrict__ fine_start,
                                                            int fshift, int N, int* __restrict__ offs, int* __restrict__ rev,
                                                            uint16_t* __restrict__ rev_bars)
{
    extern __shared__ int lds_rows[];
    __shared__ int wave_lds[kStRowsThreads / 64];
    const int R = 1 << fshift;
    int* cnt = lds_rows;
    int* stage = cnt + R;
    uint16_t* codes = reinterpret_cast<uint16_t*>(stage + kStRowsCap);
    const int b = blockIdx.x;
    const int s0 = fine_start[b], s1 = fine_start[b + 1];
    const int q0 = b << fshift;
    const int low = R - 1;
    for (int i = threadIdx.x; i < R; i += kStRowsThreads) cnt[i] = 0;
    __syncthreads();
    for (int i = s0 + (int)threadIdx.x; i < s1; i += 4 * kStRowsThreads) {
        int y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = i + u * kStRowsThreads < s1 ? rec2[i + u * kStRowsThreads].y : 0;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (i + u * kStRowsThreads < s1) atomicAdd(&cnt[y[u] & low], 1);
    }
    __syncthreads();
    int carry = 0;
    for (int c0 = 0; c0 < R; c0 += kStRowsThreads) {
        const int c = c0 + (int)threadIdx.x;
        const bool in = c < R;
        const int v = in ? cnt[c] : 0;
        int tot;
        const int ex = block_excl_scan(v, &tot, wave_lds);
        if (in) {
            cnt[c] = carry + ex;
            if (q0 + c < N) offs[q0 + c] = s0 + carry + ex;
        }
        carry += tot;
    }
    __syncthreads();
    const bool in_lds = s1 - s0 <= kStRowsCap;
    for (int i = s0 + (int)threadIdx.x; i < s1; i += 4 * kStRowsThreads) {
        int2 eq[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) eq[u] = i + u * kStRowsThreads < s1 ? rec2[i + u * kStRowsThreads] : make_int2(0, 0);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (i + u * kStRowsThreads >= s1) continue;
            const int at = atomicAdd(&cnt[eq[u].y & low], 1);
            if (in_lds) stage[at] = eq[u].x;
            else rev[s0 + at] = eq[u].x;
            if (BARS) (in_lds ? codes[at] : rev_bars[s0 + at]) = (uint16_t)((uint32_t)eq[u].y >> 16);
        }
    }
    if (in_lds) {
        __syncthreads();
        for (int i = threadIdx.x; i < s1 - s0; i += kStRowsThreads) {
            rev[s0 + i] = stage[i];
            if (BARS) rev_bars[s0 + i] = codes[i];
        }
    }
}

// ---------------------------------------------------------------------------
// The same reversed graph for medium inputs (2^21 entries and more).  k_bin_scatter sends its 8-byte records one by one to
// some thousand bins, and the lines of those stores leave the L2 before their neighbours arrive (1M x 32: 0.8 GB written
// for 0.26 GB of payload).  Here the records of a tile of 16,384 entries are sorted by bin in LDS first (their neighbours and 16-bit
// places in the tile, six bytes each), at most 1024 bins, so that a bin gets a run of 16 records (a cache line) per tile.  The rows of a bin
// are then assembled in LDS, a quarter, a half or all of its points at a time, and written whole.  (The workgroups of a bin are on different
// dies, and each reads all its records twice, from beyond the L2: 1M x 32, two of them, 0.97 GB for 0.26 GB of records at 6 TB/s.)  1M x 32: scatter 0.49 -> 0.11 ms, rows 0.26 -> 0.18; export of the graph of 100,000 x 32 182 -> 170 us, 30,000 x 100
// 241 -> 208, 50,000 x 32 the same.
constexpr int kTileThreads = 1024, kTilePer = 16, kTile = kTileThreads * kTilePer;
constexpr int kTileMaxBins = 1024;

__host__ __device__ inline size_t tile_lds_bytes(int n_bins) { return (size_t)3 * ((n_bins + 3) & ~3) * sizeof(int) + (size_t)kTile * 6; }

__global__ __launch_bounds__(kTileThreads) void k_tile_scatter(const int* __restrict__ old_idx, int total, int per_part, int N, int shift,
                                                               int n_bins, const int* __restrict__ bin_start,
                                                               const int* __restrict__ part_off, int2* __restrict__ out)
{
    extern __shared__ __align__(16) int lds_tile[];
    __shared__ int wave_lds[kTileThreads / 64];
    const int nb = (n_bins + 3) & ~3, tid = threadIdx.x;
    int* cursor = lds_tile;
    int* cnt = cursor + nb;
    int* first = cnt + nb;
    int* nbr = first + nb;
    uint16_t* place = reinterpret_cast<uint16_t*>(nbr + kTile);
    for (int b = tid; b < n_bins; b += kTileThreads) cursor[b] = bin_start[b] + part_off[(size_t)blockIdx.x * n_bins + b];
    const long long begin = (long long)blockIdx.x * per_part;
    const int e0 = (int)min((long long)total, begin), e1 = (int)min((long long)total, begin + per_part);
    const int low = (1 << shift) - 1;
    int q[kTilePer];
    auto request = [&](int t0) {
#pragma unroll
        for (int u = 0; u < kTilePer; ++u) {
            const int e = t0 + kTileThreads * u + tid;
            q[u] = e < e1 ? old_idx[e] : -1;
        }
    };
    request(e0);
    for (int t0 = e0; t0 < e1; t0 += kTile) {
        if (tid < n_bins) cnt[tid] = 0;
        __syncthreads();
        int rank[kTilePer];
#pragma unroll
        for (int u = 0; u < kTilePer; ++u) {
            if ((unsigned)q[u] >= (unsigned)N) q[u] = -1;
            rank[u] = q[u] >= 0 ? atomicAdd(&cnt[q[u] >> shift], 1) : 0;
        }
        __syncthreads();
        int n_tile;
        const int ex = block_excl_scan(tid < n_bins ? cnt[tid] : 0, &n_tile, wave_lds);
        if (tid < n_bins) first[tid] = ex;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kTilePer; ++u) {
            if (q[u] < 0) continue;
            const int at = first[q[u] >> shift] + rank[u];
            nbr[at] = q[u];
            place[at] = (uint16_t)(kTileThreads * u + tid);
        }
        __syncthreads();
        if (t0 + kTile < e1) request(t0 + kTile);
        for (int i = tid; i < n_tile; i += kTileThreads) {
            const int x = nbr[i], b = x >> shift;
            out[(size_t)cursor[b] + (size_t)(i - first[b])] = make_int2(t0 + (int)place[i], x & low);
        }
        __syncthreads();
        if (tid < n_bins) cursor[tid] += cnt[tid];
        __syncthreads();
    }
}

// Workgroup blockIdx.x: points [s 2^fshift, (s + 1) 2^fshift) of bin b, blockIdx.x = b 2^(shift - fshift) + s.
// LDS: cnt[2^fshift] | stage[kStRowsCap].
__global__ __launch_bounds__(kTileThreads) void k_tile_rows(const int2* __restrict__ rec, const int* __restrict__ bin_start, int shift,
                                                            int fshift, int N, int* __restrict__ offs, int* __restrict__ rev)
{
    extern __shared__ int lds_rows[];
    __shared__ int wave_lds[kTileThreads / 64];
    __shared__ int before_s;
    const int R = 1 << fshift, tid = threadIdx.x;
    int* cnt = lds_rows;
    int* stage = cnt + R;
    const int b = (int)blockIdx.x >> (shift - fshift), s = (int)blockIdx.x & ((1 << (shift - fshift)) - 1);
    const int s0 = bin_start[b], s1 = bin_start[b + 1];
    const int q0 = (b << shift) + (s << fshift);
    if (q0 >= N) return;
    for (int i = tid; i < R; i += kTileThreads) cnt[i] = 0;
    if (tid == 0) before_s = 0;
    __syncthreads();
    int before = 0;
    for (int i = s0 + tid; i < s1; i += 4 * kTileThreads) {
        int y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) y[u] = i + u * kTileThreads < s1 ? rec[i + u * kTileThreads].y : 0x7fffffff;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int sub = y[u] >> fshift;
            if (sub == s) atomicAdd(&cnt[y[u] & (R - 1)], 1);
            before += sub < s ? 1 : 0;
        }
    }
    before = wave_sum_i(before);
    if ((tid & 63) == 0 && before) atomicAdd(&before_s, before);
    __syncthreads();
    const int first = s0 + before_s;
    int n = 0;
    for (int c0 = 0; c0 < R; c0 += kTileThreads) {
        const int c = c0 + tid;
        const bool in = c < R;
        int tot;
        const int ex = block_excl_scan(in ? cnt[c] : 0, &tot, wave_lds);
        if (in) {
            cnt[c] = n + ex;
            if (q0 + c < N) offs[q0 + c] = first + n + ex;
        }
        n += tot;
    }
    __syncthreads();
    const bool in_lds = n <= kStRowsCap;
    for (int i = s0 + tid; i < s1; i += 4 * kTileThreads) {
        int2 r[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) r[u] = i + u * kTileThreads < s1 ? rec[i + u * kTileThreads] : make_int2(0, 0x7fffffff);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (r[u].y >> fshift != s) continue;
            const int at = atomicAdd(&cnt[r[u].y & (R - 1)], 1);
            if (in_lds) stage[at] = r[u].x;
            else rev[first + at] = r[u].x;
        }
    }
    if (in_lds) {
        __syncthreads();
        for (int i = tid; i < n; i += kTileThreads) rev[first + i] = stage[i];
    }
}

// The marks of graphs of 2^26 entries and more (those of the staged builder) with up to 32 neighbours.  A word stored somewhere in an array
// beyond the last cache is a memory write of its own, about 26 G a second whatever else goes on, and the join of 10M x 32 stored 256 M of them.
// It now writes its words in the order of R, whole lines, and they go to their places as the entries came: sorted by window of 2^21 words, 8192 words at a time in LDS, leaving as records (entry, word) in runs, each window's share reserved by one
// addition per tile and window; the same again inside a window to pieces of 2^14 words; a piece is put together in LDS and written whole, with the zeros.
// 10M x 32: join 21.96 -> 15.54 ms, the three steps 1.22 + 1.23 + 0.63, and 0.24 less for words not cleared.  (One sort by windows of 2^19 words
// and stores from there, although they meet in the L2: 1.76 + 3.04, by 2^21 1.21 + 3.54.)  Smaller graphs: 1M x 100, whose words fit the last cache, 2.85 ms of which 0.47 are the stores; the steps would
// take 0.3 of that.
constexpr int kMarkThreads = 512, kMarkPer = 16, kMarkTile = kMarkThreads * kMarkPer;
constexpr int kMarkWindow = 21, kMarkPiece = 14;          // bits

__host__ __device__ inline size_t mark_lds_bytes(int n_bins) { return (size_t)3 * ((n_bins + 3) & ~3) * sizeof(int) + (size_t)kMarkTile * sizeof(int2); }
inline int mark_windows(size_t total) { return (int)((total - 1) >> kMarkWindow) + 1; }
// counters: a line for each window, an int for each piece
inline size_t mark_ints(size_t total) { return (size_t)mark_windows(total) * (32 + ((size_t)1 << (kMarkWindow - kMarkPiece))); }

// FIRST: word i of marks belongs to entry rev[i], i < *n_in, and goes to its window; otherwise the records of window blockIdx.y (n_in[32 y] of them) to
// their pieces.  taken[stride b]: words of bin b so far (zero before the launch).  Record i of bin b of out: one of its words, in no order.
template <bool FIRST>
__global__ __launch_bounds__(kMarkThreads) void k_mark_scatter(const int* __restrict__ rev, const uint32_t* __restrict__ marks,
                                                               const int2* __restrict__ rec, const int* __restrict__ n_in, int n_bins,
                                                               int stride, int* __restrict__ taken, int2* __restrict__ out)
{
    constexpr int kBits = FIRST ? kMarkWindow : kMarkPiece;
    extern __shared__ __align__(16) int lds_mark[];
    __shared__ int wave_lds[kMarkThreads / 64];
    const int nb = (n_bins + 3) & ~3, tid = threadIdx.x;
    int* cnt = lds_mark;
    int* first = cnt + nb;
    int* base = first + nb;
    int2* stage = reinterpret_cast<int2*>(base + nb);
    if (!FIRST) {
        rec += (size_t)blockIdx.y << kMarkWindow;
        out += (size_t)blockIdx.y << kMarkWindow;
        taken += (size_t)blockIdx.y * (size_t)n_bins;
    }
    const size_t n = (size_t)(FIRST ? *n_in : n_in[32 * blockIdx.y]), step = (size_t)gridDim.x * kMarkTile;
    const int low = FIRST ? 0x7fffffff : (1 << kMarkWindow) - 1;
    int2 r[kMarkPer];
    auto request = [&](size_t t0) {
#pragma unroll
        for (int u = 0; u < kMarkPer; ++u) {
            const size_t i = t0 + (size_t)(kMarkThreads * u + tid);
            r[u] = make_int2(0, 0);
            if (FIRST && i < n) r[u] = make_int2(rev[i], (int)marks[i]);
            if (!FIRST && i < n) r[u] = rec[i];
        }
    };
    const size_t t_first = (size_t)blockIdx.x * kMarkTile;
    request(t_first);
    for (size_t t0 = t_first; t0 < n; t0 += step) {
        for (int b = tid; b < n_bins; b += kMarkThreads) cnt[b] = 0;
        __syncthreads();
        int rank[kMarkPer];
#pragma unroll
        for (int u = 0; u < kMarkPer; ++u) rank[u] = r[u].y ? atomicAdd(&cnt[(r[u].x & low) >> kBits], 1) : 0;
        __syncthreads();
        // (at most 1024 bins: two per thread)
        const int b0 = 2 * tid, c0 = b0 < n_bins ? cnt[b0] : 0, c1 = b0 + 1 < n_bins ? cnt[b0 + 1] : 0;
        if (c0) base[b0] = atomicAdd(&taken[stride * b0], c0);
        if (c1) base[b0 + 1] = atomicAdd(&taken[stride * (b0 + 1)], c1);
        int n_tile;
        const int ex = block_excl_scan(c0 + c1, &n_tile, wave_lds);
        if (b0 < n_bins) first[b0] = ex;
        if (b0 + 1 < n_bins) first[b0 + 1] = ex + c0;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kMarkPer; ++u)
            if (r[u].y) stage[first[(r[u].x & low) >> kBits] + rank[u]] = r[u];
        __syncthreads();
        if (t0 + step < n) request(t0 + step);
        for (int i = tid; i < n_tile; i += kMarkThreads) {
            const int2 x = stage[i];
            const int b = (x.x & low) >> kBits;
            out[((size_t)b << kBits) + (size_t)(base[b] + i - first[b])] = x;
        }
        __syncthreads();
    }
}

// One workgroup per piece: its words, taken[blockIdx.x] of them in records, and zeros.
__global__ __launch_bounds__(kMarkThreads) void k_mark_place(const int2* __restrict__ rec, const int* __restrict__ taken, size_t total,
                                                             uint32_t* __restrict__ pass)
{
    extern __shared__ __align__(16) int lds_mark[];
    uint4* words = reinterpret_cast<uint4*>(lds_mark);
    const size_t first = (size_t)blockIdx.x << kMarkPiece;
    const int n = taken[blockIdx.x], tid = threadIdx.x;
    rec += first;
    pass += first;
    int2 r[8];
    auto request = [&](int i) {
#pragma unroll
        for (int u = 0; u < 8; ++u) r[u] = i + kMarkThreads * u < n ? rec[i + kMarkThreads * u] : make_int2(-1, 0);
    };
    request(tid);
    for (int i = tid; i < (1 << kMarkPiece) / 4; i += kMarkThreads) words[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    for (int i = tid; i < n; i += 8 * kMarkThreads) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (r[u].x >= 0) lds_mark[r[u].x & ((1 << kMarkPiece) - 1)] = r[u].y;
        if (i + 8 * kMarkThreads < n) request(i + 8 * kMarkThreads);
    }
    __syncthreads();
    const int there = (int)min((size_t)1 << kMarkPiece, total - first);
    for (int i = tid; i < there / 4; i += kMarkThreads) reinterpret_cast<uint4*>(pass)[i] = words[i];
    if (tid < (there & 3)) pass[(there & ~3) + tid] = (uint32_t)lds_mark[(there & ~3) + tid];
}

__global__ __launch_bounds__(256) void k_mark_clear(int* __restrict__ taken, int n)
{
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b < n) taken[b] = 0;
}

// The bar of a point: s sqrt(last slot of its row / (1 - gamma)) + e_p.
// A sum bar + e_c is at least 1 + 2^-21 times the sum of the values it stands for, which covers the roundings of the sum, its square
// and the comparison.  1e-30 under the root covers what underflow takes from the chain.  An infinite or NaN last slot makes the bar
// infinite or NaN, a row that is not finite makes d~ - E1 NaN, and a comparison with that drops nothing.
// The last workgroup has no points: it takes the largest norm and error of any finite row from the parts of them (join_copy.hip).
// The others also clear the marks (words of them, none where they are put together: k_mark_place): the join stores the words that are not zero only.  A word stored somewhere in a large array is a
// memory write of its own, twice the time of a line read (26 G a second; 87 G while the array fits the last cache).
// And they take the snapshot of the neighbours: a launch less per pass (10M x 32 0.80 -> 0.77 ms for both, 1M x 100 0.094 either way; 10,000 x 32 the call 579 -> 573 us).
__global__ __launch_bounds__(256) void k_join_bars(JoinCopy jc, float* __restrict__ scale, const float* __restrict__ knn_dist, int N, int K,
                                                   float one_minus_gamma, float* __restrict__ out, uint32_t* __restrict__ pass, size_t words,
                                                   const int* __restrict__ knn_idx, int* __restrict__ old_idx)
{
    if (blockIdx.x + 1 == gridDim.x) {
        __shared__ float2 part[256];
        float2 most = make_float2(0.0f, 0.0f);
#pragma unroll 8
        for (int i = threadIdx.x; i < jc.n_parts; i += 256) {
            const float2 v = jc.parts[i];
            most = make_float2(fmaxf(most.x, v.x), fmaxf(most.y, v.y));
        }
        part[threadIdx.x] = most;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if ((int)threadIdx.x < o) {
                const float2 v = part[threadIdx.x + o];
                most = make_float2(fmaxf(most.x, v.x), fmaxf(most.y, v.y));
                part[threadIdx.x] = most;
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            scale[1] = most.x;
            scale[2] = most.y * kJoinUp;
        }
        return;
    }
    {
        const size_t pieces = words >> 2, stride = (size_t)(gridDim.x - 1) * 256, first = (size_t)blockIdx.x * 256 + threadIdx.x;
        for (size_t i = first; i < pieces; i += stride) reinterpret_cast<uint4*>(pass)[i] = make_uint4(0u, 0u, 0u, 0u);
        if (first < (words & 3)) pass[4 * pieces + first] = 0u;
        const size_t ids = (size_t)N * (size_t)K;
        for (size_t i = first; i < ids >> 2; i += stride) reinterpret_cast<i32x4_a4*>(old_idx)[i] = reinterpret_cast<const i32x4_a4*>(knn_idx)[i];
        if (first < (ids & 3)) old_idx[(ids & ~(size_t)3) + first] = knn_idx[(ids & ~(size_t)3) + first];
    }
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const float tau = knn_dist[(size_t)p * K + (K - 1)];
    out[p] = (scale[0] * sqrtf(tau / one_minus_gamma + 1e-30f) + jc.errs[p]) * kJoinUp;
}

// d~ - E1 of a pair, from S = n_p + n_c and the product g of the rows
__device__ __forceinline__ float join_least(float S, float g, float kappa)
{
    return __builtin_fmaf(-kappa, S, __builtin_fmaf(-2.0f, g, S));
}

// May the pair enter row p?  Not when d~ - E1 is above w^2, w = bar_p + e, e the largest e_c of the 32 neighbours tested together; that is, when
//   g + join_reach(n_p, bar_p + e) < join_floor(n_c),   the halves of w^2 - (1 - kappa) n_p and of (1 - kappa) n_c:
// one addition and one comparison per pair where S, d~ - E1, w and its square for each took six instructions, with branches around them.  The roundings
// of both and of the sum are below 2^-23 (w^2 + S): kJoinWide, and 2^-19 more for kappa.  (True when anything is NaN; a tie at the last
// slot may still enter: smaller index.)
constexpr float kJoinWide = 1.0f + 1.0f / 1048576.0f;
__device__ __forceinline__ float join_reach(float n_p, float w, float kappa)
{
    return 0.5f * __builtin_fmaf(kappa + 1.0f / 524288.0f - 1.0f, n_p, w * w * kJoinWide);
}
__device__ __forceinline__ float join_floor(float n_c, float kappa) { return 0.5f * (1.0f - (kappa + 1.0f / 524288.0f)) * n_c; }

// The marks of a tile of 32 points: accumulator i of lane l holds point m = 4 (l / 32) + 8 (i / 4) + i % 4 of the tile and neighbour l % 32, so the
// ballot over the wavefront holds the 32-bit masks of two points, low half for m = 8 (i / 4) + i % 4, high half for m + 4.  Lane m < 32 is left with
// the mask of point m.  reach: join_reach of the tile's points (LDS).  No branch and no wait for LDS between the sixteen, and a mask goes to its lane in
// one instruction: 10M x 32 23.06 -> 21.96 ms, 1M x 100 3.23 -> 2.86, 123,457 x 37 with K = 45 0.443 -> 0.367, 70,000 x 784 with K = 90 5.36 -> 5.05, 1M x 256
// (whose codes are stored pair by pair) 7.0 either way.  (write_lane_u32 is declared by the name of the compiler's intrinsic: with a compiler that names it otherwise
// the library does not link, for want of that symbol.)
__device__ __forceinline__ uint32_t join_masks(const f32x16& g, const float* reach, int mbase, float floor_c)
{
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
        const float4 r = *reinterpret_cast<const float4*>(reach + mbase + 2 * i);
        const float at[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint64_t bm = ballot64(!(g[i + j] + at[j] < floor_c));
            mine = write_lane_u32((uint32_t)bm, 2 * i + j, mine);
            mine = write_lane_u32((uint32_t)(bm >> 32), 2 * i + j + 4, mine);
        }
    }
    return mine;
}

// In place of the norm of a point whose pairs are not marked: above the square of any bar of a full row
// (the finite rows' coordinates are below 2^15), and no sum with it overflows.
constexpr float kNever = 1e37f;

// Where a point is among the neighbours of q, if it is: a table in LDS by the low bits of the ids, in which a later neighbour hides an
// earlier one (a mark too many, which the merge drops).
template <int SIZE>
struct JoinSelf {
    uint8_t* at;
    __device__ __forceinline__ void put(int c, int col) const { if (c >= 0) at[c & (SIZE - 1)] = (uint8_t)col; }
    __device__ __forceinline__ int find(int p) const { return at[p & (SIZE - 1)]; }     // (a column that may hold p, to be compared)
};

// One wavefront per q.  Per-wavefront LDS (ints): cq[KP] | pid[32] | reach[32] | pn[32] | perr[32] | pper[32] | pe[32] | self[64] | LINES: rows[2][32] of 128 bytes, KP = K rounded up to 32.
// Workgroups (x, y): every gridDim.y-th tile of R(q), the y-th first.
// LINES: rows through LDS.  A lane that loads its 16 bytes of a row by itself asks for a line eight times, and the address units were busy 79 % of the
// time (1M x 256; 52 % by lines); lines loaded whole cost a wavefront per SIMD and its LDS.  1M x 256 7.0 -> 6.57 ms, 100,000 x 784 1.97 -> 1.70, 60,000 x 200 with K = 130 5.3 -> 4.6, 20,000 x 300
// with K = 250 7.4 -> 5.3 (the rule and both its sides are at the launch).
template <int WAVES, bool BOUNDS, bool LINES>
__global__ __launch_bounds__(64 * WAVES, LINES ? 4 : 5) void k_explore_join(JoinCopy jc, int N, int K, const int* __restrict__ old_idx,
                                                              const float* __restrict__ bars,
                                                              const int* __restrict__ offs, const int* __restrict__ rev,
                                                              uint32_t* __restrict__ pass, uint16_t* __restrict__ bounds, int KP, int bpitch, int ksteps,
                                                              float kappa, float any_rel, float any_abs, int wave_lds_ints,
                                                              uint32_t div_m, int div_s, const int* __restrict__ order)
{
    extern __shared__ __align__(16) int lds_join[];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = die_local_place(blockIdx.x, gridDim.x) * WAVES + wave;
    if (item >= N) return;                                // whole wavefront leaves together
    const int q = order ? order[item] : item;
    const int r0 = offs[q], R = offs[q + 1] - r0;
    if (R <= 32 * (int)blockIdx.y) return;
    int* cq = lds_join + (size_t)wave * (size_t)wave_lds_ints;
    int* pid = cq + KP;
    float* reach = reinterpret_cast<float*>(pid + 32);
    float* pn = reach + 32;
    float* perr = pn + 32;
    float* pper = perr + 32;
    int* pe = reinterpret_cast<int*>(pper + 32);
    const JoinSelf<256> self{reinterpret_cast<uint8_t*>(pe + 32)};
    u32x4* rows = reinterpret_cast<u32x4*>(pe + 32 + 64);
    const int MW = KP >> 5;
    const float most_norm = jc.mu[jc.D + 1], most_err = jc.mu[jc.D + 2];

    for (int k = lane; k < KP; k += 64) {
        int c = k < K ? old_idx[(size_t)q * K + k] : -1;
        if (c < 0 || c >= N) c = -1;
        cq[k] = c;
        self.put(c, k);
    }

    for (int pt0 = 32 * (int)blockIdx.y; pt0 < R; pt0 += 32 * (int)gridDim.y) {
        const int np = min(32, R - pt0);
        wave_lds_sync();                                  // reads of the previous tile are done (and cq is written)
        int my_e = -1;                                    // lanes 0..31: the graph entry (p, k) with q = neighbour k of p
        float pbar = 0.0f;
        if (lane < 32) {
            my_e = lane < np ? rev[(size_t)r0 + pt0 + lane] : -1;
            const int p = my_e >= 0 ? (int)(((uint64_t)div_m * (uint64_t)(uint32_t)my_e) >> div_s) : -1;
            pid[lane] = p;
            pe[lane] = my_e;
            if (p >= 0) pbar = bars[p];
            if (BOUNDS) pper[lane] = 65534.0f / join_span(pbar, most_norm);
        }
        wave_lds_sync();

        const int pm = pid[lane & 31];
        const int own = pm >= 0 ? self.find(pm) % KP : 0, own_at = cq[own] == pm ? own : -1;    // place of p among the neighbours
        const int mbase = 4 * (lane >> 5);
        for (int ct = 0; ct < MW; ++ct) {
            const int cid = cq[ct * 32 + (lane & 31)];
            const uint16_t* ra = jc.rows + (size_t)(pm >= 0 ? pm : q) * (size_t)bpitch + 8 * (lane >> 5);
            const uint16_t* rb = jc.rows + (size_t)(cid >= 0 ? cid : q) * (size_t)bpitch + 8 * (lane >> 5);
            // LINES: 64 dimensions of the rows of the tile's points and of these neighbours at a time, eight lanes per row, whole lines (piece d of row r in
            // place d ^ r % 8: eight lanes that read the same piece of eight rows meet no bank twice); the next 64 travel while the products are made
            int id[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!LINES) break;
                id[i] = i < 4 ? pid[8 * i + (lane >> 3)] : cq[ct * 32 + 8 * (i - 4) + (lane >> 3)];
                if (id[i] < 0) id[i] = q;
            }
            const int at = 8 * ((lane & 7) ^ (lane >> 3));
            const auto fetch = [&](int k0) {
                if (16 * k0 + at < bpitch) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) load_to_lds(jc.rows + (size_t)id[i] * (size_t)bpitch + 16 * k0 + at, rows + 64 * i);
                }
            };
            float an = 0.0f, cn = 0.0f;                   // norms of the row of point l % 32 of the tile and of neighbour l % 32
            f32x16 g;
#pragma unroll
            for (int i = 0; i < 16; ++i) g[i] = 0.0f;
            if (LINES) {
                wave_lds_drain();
                fetch(0);
            }
            for (int k0 = 0; k0 < ksteps; k0 += 4) {
                f16x8 a[4], b[4];
                if (LINES) wave_vm_drain();
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (LINES) {
                        const int from = 8 * (lane & 31) + ((2 * u + (lane >> 5)) ^ (lane & 7));
                        a[u] = *reinterpret_cast<const f16x8*>(rows + from);
                        b[u] = *reinterpret_cast<const f16x8*>(rows + 256 + from);
                    } else if (k0 + u < ksteps) {
                        a[u] = *reinterpret_cast<const f16x8*>(ra + 16 * (k0 + u));
                        b[u] = *reinterpret_cast<const f16x8*>(rb + 16 * (k0 + u));
                    }
                }
                if (LINES) {
                    wave_lds_drain();
                    if (k0 + 4 < ksteps) fetch(k0 + 4);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (k0 + u < ksteps) {
                        g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[u], b[u], g, 0, 0, 0);
                        an = half_norm(a[u], an);
                        cn = half_norm(b[u], cn);
                    }
                }
            }
            an += __shfl_xor(an, 32, 64);
            cn += __shfl_xor(cn, 32, 64);
            const float ce = join_err(cn, any_rel, any_abs, most_err);
            const float e = wave_max(cid >= 0 ? ce : 0.0f);
            if (cid == q) cn = kNever;
            wave_lds_sync();
            if (lane < 32) {
                const float n_p = pm == q ? kNever : an;
                reach[lane] = join_reach(n_p, pbar + e, kappa);
                if (BOUNDS) {
                    pn[lane] = n_p;
                    perr[lane] = join_err(an, any_rel, any_abs, most_err);
                }
            }
            wave_lds_sync();
            const float floor_c = join_floor(cn, kappa);
            uint32_t mine = join_masks(g, reach, mbase, floor_c) & (uint32_t)ballot64(cid >= 0);   // mask of the point this lane stores (lanes 0..31)
            if (BOUNDS && cid >= 0) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int m = mbase + 8 * (i >> 2) + (i & 3);
                    if (m < np && !(g[i] + reach[m] < floor_c))
                        bounds[(size_t)pe[m] * (size_t)KP + ct * 32 + (lane & 31)] =
                            (uint16_t)join_code(join_least(pn[m] + cn, g[i], kappa), perr[m], ce, pper[m]);
                    if ((i & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // four at a time (registers)
                }
            }
            if ((own_at >> 5) == ct) mine &= ~(1u << (own_at & 31));
            if (lane < np && mine) pass[(size_t)my_e * MW + ct] = mine;
        }
    }
}

// The join for points of at most 128 dimensions where no codes are kept (KS = steps of 16 dimensions, fixed
// at compile time: 2, 4 or 8).  A wavefront takes 32 neighbours of q, one word of marks per graph entry; MANY: rows of more than 32
// neighbours, MW wavefronts beside each other for a q, which find its tiles in the caches.  The rows of the neighbours are loaded once
// and stay in registers for all tiles of R(q); the norm and last slot of the points of a tile travel while their rows
// are fetched.  A wavefront then has three dependent trips to memory per q (row offsets and neighbours | their rows
// and the elements of R(q) | the rows of those points) instead of five, and short rows leave room for twice the
// wavefronts per SIMD.  With more than 32 dimensions the rows come by whole lines through LDS (as in k_explore_join: the address units were busy 72 % of the time
// at 100 dimensions): 123,457 x 37, K = 45 0.367 -> 0.287 ms, 400,000 x 64 0.78 -> 0.59, 400,000 x 48, K = 60 1.80 -> 1.37, 200,000 x 100, K = 48 1.19 -> 0.96, 1M x
// 100 2.86 -> 2.79; 10M x 32, which is at the rate of its lines, 12.0 -> 13.1 with a wavefront per SIMD less.  The bound is that of k_explore_join.  (Against it: 1M x 100, K = 48 a
// pass 39.6 -> 37.9 ms, 1M x 24, K = 36 7.63 -> 7.39, 123,457 x 37, K = 45 1.49 -> 1.44.)
template <int WAVES, int KS, bool MANY>
__global__ __launch_bounds__(64 * WAVES, KS == 4 ? 7 : 1) void k_explore_join_short(JoinCopy jc, int N, int K, const int* __restrict__ old_idx,
                                                                    const float* __restrict__ bars,
                                                                    const int* __restrict__ offs, const int* __restrict__ rev,
                                                                    const uint16_t* __restrict__ rev_bars,
                                                                    uint32_t* __restrict__ pass, uint32_t* __restrict__ marks, int MW, int bpitch, int ksteps,
                                                                    float kappa, float any_rel, float any_abs, uint32_t div_m, int div_s,
                                                                    const int* __restrict__ order)
{
    constexpr bool LINES = KS > 2;
    constexpr int P = 2 * KS;                             // 16-byte pieces of a row in LDS
    __shared__ u32x4 rows_s[WAVES][LINES ? 32 * P : 1];
    __shared__ int pid_s[WAVES][32];
    __shared__ __align__(16) float reach_s[WAVES][32];
    __shared__ uint8_t self_s[WAVES][128];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int unit = __builtin_amdgcn_readfirstlane(die_local_place(blockIdx.x, gridDim.x) * WAVES + wave);
    const int item = MANY ? (int)((unsigned)unit / (unsigned)MW) : unit, ct = MANY ? unit - item * MW : 0;
    if (item >= N) return;                                // whole wavefront leaves together
    const int q = order ? order[item] : item;
    const int r0 = offs[q], R = offs[q + 1] - r0;
    const int col = lane & 31, hi = lane >> 5;
    int cid = 32 * ct + col < K ? old_idx[(size_t)q * K + 32 * ct + col] : -1;
    if (R <= 32 * (int)blockIdx.y) return;
    if (cid < 0 || cid >= N) cid = -1;
    int* pid = pid_s[wave];
    u32x4* rows = rows_s[wave];
    // LINES: the rows of the points in pid go to LDS, whole lines at a time (P lanes per row, KS loads): piece d of row r in place d ^ r % 8, so that eight
    // lanes that read the same piece of eight rows meet no bank twice.
    const auto fetch = [&]() {
#pragma unroll
        for (int i = 0; i < KS; ++i) {
            const int r = (64 / P) * i + lane / P, piece = (lane % P) ^ (r & 7), id = pid[r];
            if (KS <= 4 || 8 * piece < bpitch) load_to_lds(jc.rows + (size_t)(id >= 0 ? id : q) * (size_t)bpitch + 8 * piece, rows + 64 * i);
        }
    };
    const auto from_lds = [&](int u) { return *reinterpret_cast<const f16x8*>(rows + col * P + ((2 * u + hi) ^ (col & 7))); };
    const uint16_t* rb = jc.rows + (size_t)(cid >= 0 ? cid : q) * (size_t)bpitch + 8 * hi;
    if (LINES) {
        if (lane < 32) pid[lane] = cid;
        wave_lds_sync();
        fetch();
        wave_vm_drain();
    }
    f16x8 b[KS];
#pragma unroll
    for (int u = 0; u < KS; ++u) {
#pragma unroll
        for (int i = 0; i < 8; ++i) b[u][i] = (_Float16)0.0f;
        if (KS <= 4 || u < ksteps) b[u] = LINES ? from_lds(u) : *reinterpret_cast<const f16x8*>(rb + 16 * u);
    }
    float cn = 0.0f;
#pragma unroll
    for (int u = 0; u < KS; ++u) cn = half_norm(b[u], cn);
    cn += __shfl_xor(cn, 32, 64);
    const float e = wave_max(cid >= 0 ? join_err(cn, any_rel, any_abs, jc.mu[jc.D + 2]) : 0.0f);
    const float floor_c = join_floor(cid == q ? kNever : cn, kappa);
    const uint32_t there = (uint32_t)ballot64(cid >= 0);
    const JoinSelf<128> self{self_s[wave]};
    self.put(cid, col);
    const int mbase = 4 * hi;
    float* reach = reach_s[wave];

    for (int pt0 = 32 * (int)blockIdx.y; pt0 < R; pt0 += 32 * (int)gridDim.y) {
        const int np = min(32, R - pt0);
        int my_e = -1;                                    // lanes 0..31: the graph entry (p, k) with q = neighbour k of p
        float bar = 0.0f;
        if (lane < 32) {
            my_e = lane < np ? rev[(size_t)r0 + pt0 + lane] : -1;
            const int p = my_e >= 0 ? (int)(((uint64_t)div_m * (uint64_t)(uint32_t)my_e) >> div_s) : -1;
            pid[lane] = p;
            if (lane < np && rev_bars) bar = bar_of(rev_bars[(size_t)r0 + pt0 + lane]);
            else if (p >= 0) bar = bars[p];
        }
        wave_lds_sync();
        const int pm = pid[col];
        const int own = pm >= 0 ? self.find(pm) & 31 : 0;
        const bool own_there = __shfl(cid, own, 64) == pm && pm >= 0;                       // p is neighbour `own` of these
        const uint16_t* ra = jc.rows + (size_t)(pm >= 0 ? pm : q) * (size_t)bpitch + 8 * hi;
        if (LINES) {
            wave_lds_drain();                             // (the rows before have been read)
            fetch();
            wave_vm_drain();
        }
        f32x16 g;
#pragma unroll
        for (int i = 0; i < 16; ++i) g[i] = 0.0f;
        float an = 0.0f;
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            if (KS <= 4 || u < ksteps) {
                const f16x8 a = LINES ? from_lds(u) : *reinterpret_cast<const f16x8*>(ra + 16 * u);
                g = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[u], g, 0, 0, 0);
                an = half_norm(a, an);
            }
            if ((u & 1) == 1) __builtin_amdgcn_sched_barrier(0);       // two steps at a time (registers)
        }
        an += __shfl_xor(an, 32, 64);
        if (lane < 32) reach[lane] = join_reach(pm == q ? kNever : an, bar + e, kappa);
        wave_lds_sync();
        uint32_t mine = join_masks(g, reach, mbase, floor_c) & there;    // mask of the point this lane stores (lanes 0..31)
        if (own_there) mine &= ~(1u << own);
        if (!MANY && marks) {
            if (lane < np) marks[(size_t)r0 + pt0 + lane] = mine;          // (in the order of R: k_mark_scatter)
        } else if (lane < np && mine) pass[MANY ? (size_t)my_e * (size_t)MW + (size_t)ct : (size_t)my_e] = mine;
        wave_lds_sync();                                  // the tile's LDS values are read before the next tile writes them
    }
}

// The join with one workgroup (four wavefronts) per q, for rows of more than 32 neighbours.  k_explore_join loads the rows of a tile of R(q) again for every group of 32 neighbours and the rows of
// the neighbours again for every tile of R(q): at K = 90 (three groups, three tiles) every row three times.  Here 96
// points of R(q) and all neighbours of q pass through LDS together, 64 dimensions at a time (the next 64 are requested
// while these are used), and the wavefronts share the pairs (tile of R(q), group of neighbours) among them, each
// keeping the accumulators of its pairs: every row is read once per 96 points of R(q).  Bound and outputs are those
// of k_explore_join.  NPW = pairs per wavefront (3: K <= 128, at three wavefronts per SIMD, 70,000 x 784, K = 90 6.9 -> 5.1 ms against two; 6: K <= 256, at
// one).
constexpr int kJwP = 96;                    // points of R(q) worked on together (three tiles)
constexpr int kJwRowBytes = 144;            // 64 float16 values + 16 bytes: rows start in different banks

template <bool BOUNDS, int NPW>
__global__ __launch_bounds__(256, NPW == 3 ? 3 : 1) void k_explore_join_wg(JoinCopy jc, int N, int K, const int* __restrict__ old_idx,
                                                         const float* __restrict__ bars, const int* __restrict__ offs,
                                                         const int* __restrict__ rev, uint32_t* __restrict__ pass,
                                                         uint16_t* __restrict__ bounds, int KP, int bpitch, int ksteps,
                                                         float kappa, float any_rel, float any_abs, uint32_t div_m, int div_s,
                                                         const int* __restrict__ order)
{
    constexpr int kPieces = (kJwP + (NPW == 3 ? 128 : 256)) * 8 / 256;     // 16-byte pieces a thread stages per step
    extern __shared__ __align__(16) unsigned char lds_jw[];
    __shared__ uint8_t self_s[512];
    __shared__ float wave_e[4];
    unsigned char* rowsb = lds_jw;                                         // kJwP + KP rows of 144 bytes
    int* cq = reinterpret_cast<int*>(rowsb + (size_t)(kJwP + KP) * kJwRowBytes);
    float* cn = reinterpret_cast<float*>(cq + KP);
    float* cerr = cn + KP;
    int* pid = reinterpret_cast<int*>(cerr + KP);
    int* pe = pid + kJwP;
    float* pn = reinterpret_cast<float*>(pe + kJwP);
    float* reach = pn + kJwP;
    float* perr = reach + kJwP;
    float* pper = perr + kJwP;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 31, h = lane >> 5;
    const int item = die_local_place(blockIdx.x, gridDim.x);
    if (item >= N) return;                                                 // the whole workgroup leaves together
    const int q = order ? order[item] : item;
    const int r0 = offs[q], R = offs[q + 1] - r0;
    if (R <= kJwP * (int)blockIdx.y) return;
    const int MW = KP >> 5;
    const int nrows = kJwP + KP;
    const float most_norm = jc.mu[jc.D + 1], most_err = jc.mu[jc.D + 2];
    const JoinSelf<512> self{self_s};
    float e_most = 0.0f;                                                   // the largest e_c of all the neighbours
    for (int k = tid; k < KP; k += 256) {
        int c = k < K ? old_idx[(size_t)q * K + k] : -1;
        if (c < 0 || c >= N) c = -1;
        cq[k] = c;
        const float n_c = c >= 0 ? jc.norms[c] : 0.0f;
        self.put(c, k);
        cn[k] = c == q ? kNever : n_c;
        const float ce = join_err(n_c, any_rel, any_abs, most_err);
        cerr[k] = ce;
        if (c >= 0) e_most = fmaxf(e_most, ce);
    }
    e_most = wave_max(e_most);
    if (lane == 0) wave_e[wave] = e_most;
    __syncthreads();
    e_most = fmaxf(fmaxf(wave_e[0], wave_e[1]), fmaxf(wave_e[2], wave_e[3]));
    for (int pg = kJwP * (int)blockIdx.y; pg < R; pg += kJwP * (int)gridDim.y) {
        const int npg = min(kJwP, R - pg);
        const int npairs = ((npg + 31) >> 5) * MW;
        __syncthreads();                                                   // the previous group is done with the LDS
        if (tid < kJwP) {
            const int e = tid < npg ? rev[(size_t)r0 + pg + tid] : -1;
            const int p = e >= 0 ? (int)(((uint64_t)div_m * (uint64_t)(uint32_t)e) >> div_s) : -1;
            const float n_p = p >= 0 ? jc.norms[p] : 0.0f, bar = p >= 0 ? bars[p] : 0.0f;
            pid[tid] = p;
            pe[tid] = e;
            const float n_m = p == q ? kNever : n_p;
            pn[tid] = n_m;
            reach[tid] = join_reach(n_m, bar + e_most, kappa);
            if (BOUNDS) {
                perr[tid] = join_err(n_p, any_rel, any_abs, most_err);
                pper[tid] = 65534.0f / join_span(bar, most_norm);
            }
        }
        __syncthreads();
        f32x16 acc[NPW];
#pragma unroll
        for (int i = 0; i < NPW; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[i][j] = 0.0f;
        // pieces this thread stages: piece i = tid + 256 j of the (row, 16-byte piece) grid
        uint4 pre[kPieces];
        auto request = [&](int c0) {
#pragma unroll
            for (int j = 0; j < kPieces; ++j) {
                const int i = tid + 256 * j;
                pre[j] = make_uint4(0u, 0u, 0u, 0u);
                if (i < nrows * 8) {
                    const int r = i >> 3, pc = i & 7;
                    const int id = r < kJwP ? pid[r] : cq[r - kJwP];
                    const int el = c0 * 16 + pc * 8;
                    if (id >= 0 && el < ksteps * 16)
                        pre[j] = *reinterpret_cast<const uint4*>(jc.rows + (size_t)id * (size_t)bpitch + el);
                }
            }
        };
        request(0);
        for (int c0 = 0; c0 < ksteps; c0 += 4) {
            if (c0 > 0) __syncthreads();                                   // the previous step's values have been used
#pragma unroll
            for (int j = 0; j < kPieces; ++j) {
                const int i = tid + 256 * j;
                if (i < nrows * 8) *reinterpret_cast<uint4*>(rowsb + (size_t)(i >> 3) * kJwRowBytes + (i & 7) * 16) = pre[j];
            }
            __syncthreads();
            if (c0 + 4 < ksteps) request(c0 + 4);
#pragma unroll
            for (int i = 0; i < NPW; ++i) {
                const int pair = wave + 4 * i;
                if (pair < npairs) {
                    const int pt = pair / MW, ct = pair - pt * MW;
                    const unsigned char* ra = rowsb + (size_t)(pt * 32 + n) * kJwRowBytes + h * 16;
                    const unsigned char* rb = rowsb + (size_t)(kJwP + ct * 32 + n) * kJwRowBytes + h * 16;
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (c0 + u < ksteps) {
                            const f16x8 a = *reinterpret_cast<const f16x8*>(ra + 32 * u);
                            const f16x8 b = *reinterpret_cast<const f16x8*>(rb + 32 * u);
                            acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[i], 0, 0, 0);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);                         // one pair after the other (registers)
            }
        }
        // Accumulator j of lane l: point 4 (l / 32) + 8 (j / 4) + j % 4 of the tile, column = neighbour l % 32 of the group.
#pragma unroll
        for (int i = 0; i < NPW; ++i) {
            const int pair = wave + 4 * i;
            if (pair < npairs) {
                const int pt = pair / MW, ct = pair - pt * MW;
                const int col = ct * 32 + n;
                const int cid = cq[col];
                const float cnv = cn[col], ce = cerr[col], floor_c = join_floor(cnv, kappa);
                uint32_t mine = join_masks(acc[i], reach + pt * 32, 4 * h, floor_c) & (uint32_t)ballot64(cid >= 0);
                if (BOUNDS && cid >= 0) {
#pragma unroll
                    for (int j = 0; j < 16; ++j) {
                        const int m = pt * 32 + 4 * h + 8 * (j >> 2) + (j & 3);
                        if (m < npg && !(acc[i][j] + reach[m] < floor_c))
                            bounds[(size_t)pe[m] * (size_t)KP + col] =
                                (uint16_t)join_code(join_least(pn[m] + cnv, acc[i][j], kappa), perr[m], ce, pper[m]);
                        if ((j & 3) == 3) __builtin_amdgcn_sched_barrier(0);   // four at a time (registers)
                    }
                }
                const int p = pid[pt * 32 + (lane & 31)], own = p >= 0 ? self.find(p) : 0;
                if (p >= 0 && (own >> 5) == ct && cq[own] == p) mine &= ~(1u << (own & 31));
                if (lane < 32 && pt * 32 + lane < npg && mine) pass[(size_t)pe[pt * 32 + lane] * MW + ct] = mine;
            }
        }
    }
}

}  // namespace

// The join is used unless RSFK_EXPLORE_JOIN=0 is set, K is above 256, the graph has about 2^31 or more entries or N is beyond what the
// builder of the reversed graph takes (6144 bins of 2^13 points).
bool explore_join_enabled(int N, int K)
{
    const char* env = std::getenv("RSFK_EXPLORE_JOIN");
    if (env && env[0] == '0') return false;
    if (K > kMaxKJoin) return false;          // (rows of more than 256 neighbours: the general kernel only)
    int shift, n_bins;
    return (size_t)N * (size_t)K < kMaxEntries && rev_bins(N, &shift, &n_bins);
}

int explore_ws_alloc(ExploreWorkspace** out, int N, int K, bool with_bounds, bool graph_only)
{
    *out = nullptr;
    auto* w = new ExploreWorkspace();
    w->N = N;
    w->K = K;
    w->MW = (K + 31) / 32;
    if (!rev_bins(N, &w->shift, &w->n_bins) || (size_t)N * (size_t)K >= kMaxEntries) {
        delete w;
        set_last_error("exploration workspace: graph too large for the join");
        return 1;
    }
    const size_t total = (size_t)N * (size_t)K;
    w->n_parts = (int)std::min<size_t>(512, std::max<size_t>(1, (total + 8191) / 8192));
    w->per_part = (int)(((total + w->n_parts - 1) / w->n_parts + 1023) / 1024 * 1024);
    int l = 0;
    while ((1 << l) < K) ++l;
    w->div_s = 31 + l;
    w->div_m = (uint32_t)((((uint64_t)1 << w->div_s) + (uint64_t)K - 1) / (uint64_t)K);
    // Graphs of up to 2^18 entries (RSFK_REV_STAGED=3: of up to 2^21) take the builder of one launch.
    {
        const char* e = std::getenv("RSFK_REV_STAGED");
        const int per = std::max(1, (N + 255) / 256);
        if ((e && *e ? e[0] == '3' && total <= ((size_t)1 << 21) : total <= kDirectMost) && per <= kDirectMostPer) w->direct = per;
    }
    // Graphs of 2^21 to 2^26 entries (RSFK_REV_STAGED=2: whenever the bins allow it) take the builder that sorts tiles in LDS.
    {
        const char* e = std::getenv("RSFK_REV_STAGED");
        int cs = 0, fs = 0;
        while ((((size_t)N - 1) >> cs) + 1 > (size_t)kTileMaxBins) ++cs;
        while (fs < cs && ((size_t)3 << (fs + 1)) * (size_t)K <= (size_t)2 * kStRowsCap) ++fs;     // 1.5 K 2^fs <= cap
        const bool fits = cs - fs <= 2 && ((size_t)3 << fs) * (size_t)K <= (size_t)2 * kStRowsCap;
        if (e && *e ? e[0] == '2' : total >= ((size_t)1 << 21) && total < ((size_t)1 << 26)) w->tiled = fits;
        if (w->tiled) {
            w->cshift = cs;
            w->fshift = fs;
            w->n_coarse = (int)((((size_t)N - 1) >> cs) + 1);
            w->n_bins = std::max(w->n_bins, w->n_coarse);
            w->n_parts = (int)std::min<size_t>(256, (total + kTile - 1) / kTile);
            w->per_part = (int)(((total + w->n_parts - 1) / w->n_parts + kTile - 1) / kTile * kTile);
        }
    }
    auto dm = [graph_only](void* p, size_t n) {
        const size_t bytes = std::max<size_t>(n, 1) * sizeof(int);
        void** out = reinterpret_cast<void**>(p);
        return (graph_only ? ws_try_alloc(out, bytes) : ws_alloc(out, bytes)) ? hipErrorOutOfMemory : hipSuccess;
    };
    // Large graphs (2^26 entries and more; RSFK_REV_STAGED=1|0 says otherwise) take the builder that stages its stores
    // in LDS: fine bins whose rows fit into LDS with room to spare, about as many fine bins per coarse bin as there
    // are coarse bins.
    {
        const char* e = std::getenv("RSFK_REV_STAGED");
        bool want = total >= ((size_t)1 << 26);
        if (e && e[0] == '1') want = true;
        if (e && e[0] == '0') want = false;
        if (want && !w->tiled) {
            int fs = 5;
            while (fs < 12 && ((size_t)3 << (fs + 1)) * (size_t)K <= (size_t)2 * kStRowsCap) ++fs;    // 1.5 K 2^fs <= cap
            const int n_fine = (int)(((size_t)N + ((size_t)1 << fs) - 1) >> fs);
            int lp = 4;
            while (lp < 10 && ((size_t)1 << (2 * (lp + 1))) <= (size_t)n_fine) ++lp;                   // 2^lp about sqrt(n_fine)
            while (lp < 10 && (((size_t)N - 1) >> (fs + lp)) + 1 > (size_t)kStMaxBins) ++lp;
            const int n_coarse = (int)((((size_t)N - 1) >> (fs + lp)) + 1);
            // (the parts' counters and the bins' sizes and starts are the arrays of the one-level builder)
            if (n_coarse <= kStMaxBins && n_coarse <= w->n_bins) {
                w->staged = true;
                w->fshift = fs;
                w->cshift = fs + lp;
                w->n_coarse = n_coarse;
                w->n_fine = n_coarse << lp;
                w->n_sub = (int)(total / kStSub) + n_coarse + 2;
            }
        }
    }
    if (w->staged &&
        (dm(&w->bin_eq2, 2 * total) != hipSuccess || dm(&w->fine_size, (size_t)w->n_fine) != hipSuccess ||
         dm(&w->fine_start, (size_t)w->n_fine + 1) != hipSuccess ||
         dm(&w->sub_off, std::max((size_t)w->n_sub << (w->cshift - w->fshift), mark_ints(total))) != hipSuccess)) {
        explore_ws_free(w);
        if (!graph_only) set_last_error("exploration workspace: out of device memory");
        return 1;
    }
    if (dm(&w->rev, total) != hipSuccess || dm(&w->bin_eq, 2 * total) != hipSuccess ||
        dm(&w->offs, (size_t)N + 1) != hipSuccess || dm(&w->bin_size, (size_t)w->n_bins) != hipSuccess ||
        dm(&w->bin_start, (size_t)w->n_bins + 1) != hipSuccess ||
        dm(&w->part_off, (size_t)w->n_parts * (size_t)w->n_bins) != hipSuccess || (!graph_only && (dm(&w->pass, total * w->MW) != hipSuccess || dm(&w->bars, (size_t)N) != hipSuccess)) ||
        dm(&w->todo, todo_ints(N)) != hipSuccess) {
        explore_ws_free(w);
        if (!graph_only) set_last_error("exploration workspace: out of device memory");
        return 1;
    }
    if (with_bounds) {
        // 2 bytes per pair of the join; without them the merge still works, in the order of the marks.  The array grows
        // with N K^2 (17 GB at N = 1M, K = 90): it is only asked for up to 16 GiB, and as a block the call can do
        // without (no idle block is given up for it, a refusal leaves no error text behind)
        const size_t bytes = total * w->MW * 32 * sizeof(uint16_t);
        void* b = nullptr;
        if (bytes <= ((size_t)16 << 30) && ws_try_alloc(&b, bytes) == 0) w->bounds = static_cast<uint16_t*>(b);
    }
    // The codes of the bars beside the reversed graph, in the records of the first scatter, which are done with when the rows are made.
    // Bins of more than 2^16 points leave no room in a record, rows of more than 2^11 points at a time none in LDS.
    if (!graph_only && !w->bounds && w->staged && w->cshift <= 16 && w->fshift <= 11) w->rev_bars = reinterpret_cast<uint16_t*>(w->bin_eq);
    *out = w;
    return 0;
}

void explore_ws_free(ExploreWorkspace* w)
{
    if (!w) return;
    void* bufs[] = {w->rev, w->bin_eq, w->offs, w->bin_size, w->bin_start, w->part_off, w->pass, w->bars, w->todo, w->bounds,
                    w->bin_eq2, w->fine_size, w->fine_start, w->sub_off};
    for (void* b : bufs)
        ws_free(b);
    delete w;
}

const uint32_t* explore_ws_pass(const ExploreWorkspace* w) { return w->pass; }
const JoinBounds& explore_ws_bounds(const ExploreWorkspace* w) { return w->view; }
// The shares: kTodoShares lists of todo_share(N) points, the number of each in a cache line of its own.
int* explore_ws_share_lists(ExploreWorkspace* w) { return w->todo + 2 * ((size_t)w->N + 1); }
int* explore_ws_todo(ExploreWorkspace* w, int which) { return w->todo + (size_t)which * ((size_t)w->N + 1); }

bool explore_ws_takes(int N, int K)
{
    int shift, n_bins;
    return (size_t)N * (size_t)K < kMaxEntries && rev_bins(N, &shift, &n_bins);
}
const int* explore_ws_offs(const ExploreWorkspace* w) { return w->offs; }
int* explore_ws_rev(const ExploreWorkspace* w) { return w->rev; }

namespace {

// with_bars: rev_bars too, from bars
int launch_rev(ExploreWorkspace* w, const int* old_idx, int N, int K, hipStream_t stream, bool with_bars)
{
    RSFK_CHECK(w && w->N == N && w->K == K, "reversed graph: workspace does not match");
    const int total = (int)((size_t)N * (size_t)K);
    const RevBars rb{w->bars, w->div_m, w->div_s};
    const size_t rows_lds = ((size_t)(1 << w->fshift) + kStRowsCap) * sizeof(int) + (with_bars ? kStRowsCap * sizeof(uint16_t) : 0);
    if (w->direct) {
        hipLaunchKernelGGL(k_rev_direct, dim3((unsigned)((N + w->direct - 1) / w->direct)), dim3(kDirectThreads), (size_t)w->direct * sizeof(int), stream,
                           old_idx, total, N, w->direct, w->offs, w->rev, w->todo + 2 * (size_t)N + 1, explore_ws_shares(w));
    } else if (w->staged) {
        const int nc = w->n_coarse, per = 1 << (w->cshift - w->fshift);
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, stream, w->bin_size, nc,
                           w->todo + 2 * (size_t)N + 1, explore_ws_shares(w));
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((w->n_fine + 255) / 256)), dim3(256), 0, stream, w->fine_size, w->n_fine,
                           w->todo + 2 * (size_t)N + 1, explore_ws_shares(w));
        hipLaunchKernelGGL(k_bin_count, dim3((unsigned)w->n_parts), dim3(256), (size_t)nc * sizeof(int), stream, old_idx, total,
                           w->per_part, N, w->cshift, nc, w->bin_size, w->part_off);
        hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(256), 0, stream, w->bin_size, nc, w->bin_start, w->offs + N);
        auto* scatter1 = with_bars ? k_staged_scatter1<true> : k_staged_scatter1<false>;
        hipLaunchKernelGGL(scatter1, dim3((unsigned)w->n_parts), dim3(256), staged_lds_bytes(nc), stream, old_idx, total,
                           w->per_part, N, w->cshift, nc, w->bin_start, w->part_off, w->bin_eq, rb);
        // sub-parts of a coarse bin walked by a few workgroups each (four times the mean number of sub-parts per bin)
        const unsigned walkers = (unsigned)std::max<size_t>(1, std::min<size_t>(64, 4 * ((size_t)total / kStSub / (size_t)nc + 1)));
        hipLaunchKernelGGL(k_staged_count2, dim3(walkers, (unsigned)nc), dim3(256), (size_t)per * sizeof(int), stream, w->bin_eq,
                           w->bin_start, w->cshift, w->fshift, w->fine_size, w->sub_off);
        hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(256), 0, stream, w->fine_size, w->n_fine, w->fine_start, w->offs + N);
        RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_staged_scatter2), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)staged2_lds_bytes(per)));
        hipLaunchKernelGGL(k_staged_scatter2, dim3(walkers, (unsigned)nc), dim3(kSt2Threads), staged2_lds_bytes(per), stream, w->bin_eq,
                           w->bin_start, w->cshift, w->fshift, w->fine_start, w->sub_off, w->bin_eq2);
        auto* rows = with_bars ? k_staged_rows<true> : k_staged_rows<false>;
        RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(rows), hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_lds));
        hipLaunchKernelGGL(rows, dim3((unsigned)w->n_fine), dim3(kStRowsThreads), rows_lds, stream, w->bin_eq2, w->fine_start,
                           w->fshift, N, w->offs, w->rev, w->rev_bars);
    } else if (w->tiled) {
        const int nc = w->n_coarse;
        hipLaunchKernelGGL(k_zero, dim3((unsigned)((nc + 255) / 256)), dim3(256), 0, stream, w->bin_size, nc,
                           w->todo + 2 * (size_t)N + 1, explore_ws_shares(w));
        hipLaunchKernelGGL(k_bin_count, dim3((unsigned)w->n_parts), dim3(1024), (size_t)nc * sizeof(int), stream, old_idx, total,
                           w->per_part, N, w->cshift, nc, w->bin_size, w->part_off);
        hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(256), 0, stream, w->bin_size, nc, w->bin_start, w->offs + N);
        RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_tile_scatter), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)tile_lds_bytes(nc)));
        hipLaunchKernelGGL(k_tile_scatter, dim3((unsigned)w->n_parts), dim3(kTileThreads), tile_lds_bytes(nc), stream, old_idx, total,
                           w->per_part, N, w->cshift, nc, w->bin_start, w->part_off, w->bin_eq);
        RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_tile_rows), hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_lds));
        hipLaunchKernelGGL(k_tile_rows, dim3((unsigned)(nc << (w->cshift - w->fshift))), dim3(kTileThreads), rows_lds, stream, w->bin_eq,
                           w->bin_start, w->cshift, w->fshift, N, w->offs, w->rev);
    } else {
    const int nbins = w->n_bins;
    const size_t bin_lds = (size_t)nbins * sizeof(int);
    hipLaunchKernelGGL(k_zero, dim3((unsigned)((nbins + 255) / 256)), dim3(256), 0, stream, w->bin_size, nbins,
                       w->todo + 2 * (size_t)N + 1, explore_ws_shares(w));
    hipLaunchKernelGGL(k_bin_count, dim3((unsigned)w->n_parts), dim3(256), bin_lds, stream, old_idx, total, w->per_part, N,
                       w->shift, nbins, w->bin_size, w->part_off);
    hipLaunchKernelGGL(k_bin_scan, dim3(1), dim3(256), 0, stream, w->bin_size, nbins, w->bin_start, w->offs + N);
    hipLaunchKernelGGL(k_bin_scatter, dim3((unsigned)w->n_parts), dim3(256), bin_lds, stream, old_idx, total, w->per_part, N,
                       w->shift, nbins, w->bin_start, w->part_off, w->bin_eq);
    hipLaunchKernelGGL(k_bin_rows, dim3((unsigned)nbins), dim3(kRowsBlock), sizeof(int) << w->shift, stream, w->bin_eq,
                       w->bin_start, w->shift, N, w->offs, w->rev);
    }
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace

// The reversed graph of idx (offs, rev).
int launch_reversed_graph(ExploreWorkspace* w, const int* old_idx, int N, int K, hipStream_t stream)
{
    return launch_rev(w, old_idx, N, K, stream, false);
}

// Fill pass (and bounds) from the snapshot old_idx, which is made here, and the current last slots of knn_dist (rows sorted by distance).
int launch_explore_join(ExploreWorkspace* w, const JoinCopy& jc, int N, int D, int K, const int* knn_idx, int* old_idx,
                        const float* knn_dist, hipStream_t stream, const int* order)
{
    RSFK_CHECK(w && w->N == N && w->K == K, "exploration join: workspace does not match");
    RSFK_CHECK(K >= 1 && K <= 256, "exploration join: K must be in 1..256");
    RSFK_CHECK((size_t)N * (size_t)K < kMaxEntries, "exploration join: N*K must be below 2^31 - 4096");

    constexpr int kWaves = 4;
    const int KP = (K + 31) & ~31;
    // A few points are in hundreds of rows, and a launch over few points ends with the tiles of these, one after the other: they are
    // dealt out to several wavefronts (3,000 x 200, K = 30: 0.102 ms per pass with one, 0.029 with 16; 20,000 x 32 0.037, 0.038 with 3,
    // 0.056 with 16; 1M x 256 7.0, 7.2 with 2).  Between these a part more or less weighs little, microseconds with 1, 2, 3 and 4 parts: x 32 in
    // 64 clusters 21,000 38 35 36 36, 26,000 45 42 42 44, 32,000 51 50 51 54, 45,000 67 68 73 76, 60,000 88 92 98 102; uniform x 100 21,000 70 71
    // 75 77, 32,000 96 103 110 114, 60,000 164 184 200 213.
    const unsigned parts = (unsigned)std::max(1, std::min(16, 65536 / N));
    // (k_explore_join) Whole lines through LDS or each lane its own 16 bytes: rows are fetched 64 dimensions at a time, so a last step of up to 32 costs what
    // a full one does, and with up to 32 neighbours, where rows are read once, that decides up to 288 dimensions.  Own -> lines, us: K = 32, 20,000 x 161 92 -> 97,
    // 192 96 -> 97, 208 94 -> 108, 240 113 -> 109, 272 114 -> 121, 289 137 -> 122, 600 228 -> 200; 300,000 x 160 1322 -> 1345, 176 1388 -> 1352, 208 1637 -> 1646, 256
    // 1809 -> 1688, 320 2235 -> 2011; K = 24, 1M x 176 3919 -> 4048, 224 4760 -> 4762, 256 4900 -> 4715; K = 12, 60,000 x 208 120 -> 139, 240 141 -> 139, 257 138 -> 154, 320 173 ->
    // 156.  More neighbours: K = 50, 100,000 x 144 1148 -> 1151, 161 1217 -> 1169, 200 1459 -> 1461, 20,000 x 161 221 -> 223, 192 232 -> 221, 200 239 -> 248, 288 310 -> 291;
    // K = 140, 8,000 x 130 499 -> 539, 161 601 -> 551, 224 683 -> 621.
    const bool lines = KP > 32 ? D > 160 : D > 288 || (D > 224 && D <= 256);
    const int wave_ints = KP + 256 + (lines ? 2 * 32 * 32 : 0);
    const size_t lds = (size_t)kWaves * (size_t)wave_ints * sizeof(int);
    const int ksteps = (D + 15) / 16;
    RSFK_CHECK(ksteps * 16 <= join_pitch(D), "exploration join: rows of the copy too short");
    const float kappa = (float)(ksteps * 16 + 16) * (1.0f / 2097152.0f);            // (Dp + 16) 2^-21
    const float one_minus_gamma = 1.0f - (float)(D + 8) * (1.0f / 4194304.0f);      // 1 - (D + 8) 2^-22
    RSFK_CHECK(one_minus_gamma > 0.5f, "exploration join: D too large");
    const float any_rel = join_err_rel(), any_abs = join_err_abs(D);
    w->view.codes = w->bounds;
    w->view.bars = w->bars;
    w->view.norms = jc.norms;
    w->view.scale = jc.scale();
    w->view.kappa = kappa;
    w->view.one_minus_gamma = one_minus_gamma;
    w->view.any_rel = any_rel;
    w->view.any_abs = any_abs;
    const int MW = KP >> 5;
    // More points than a launch has threads for take a wavefront per q: with a wavefront per 32 neighbours K = 33 from 33.5 million points on, 129
    // from 13.4, 225 from 8.4, with a workgroup per q all from 16.8.
    // One workgroup per q reads every row once per 96 points of R(q), one wavefront per q (and 32 neighbours) again for every group of 32
    // neighbours, so the former pays with the bytes that are read again, D (K - 24) or so, sooner with more groups; up to 32 neighbours
    // are one pair per tile of R(q), too little for four wavefronts (1M x 256, K = 32: 8.1 ms against 12.6).  A pass, a wavefront per q -> a
    // workgroup: 123,457 x 37, K = 45 1.49 -> 2.08 ms, 300,000 x 64, K = 64 10.1 -> 11.6, x 200 16.7 -> 16.8, x 300 20.0 -> 18.5, 200,000 x 600, K = 40
    // 10.9 -> 10.4, 300,000 x 64, K = 90 17.8 -> 19.0, x 100 20.8 -> 20.8, 100,000 x 128, K = 90 7.07 -> 6.89, x 400 12.3 -> 9.6, 200,000 x 16, K = 128 19.3
    // -> 19.6, x 32 17.0 -> 16.9, 100,000 x 256, K = 128 15.0 -> 11.4.  Above 128 neighbours its accumulators leave one wavefront per SIMD, and the
    // line is far up: 8,000 points after one tree, x 400, K = 256 21.33 -> 21.38, x 550, K = 190 14.04 -> 13.99, K = 220 18.1 -> 17.7, x 784, K = 130 8.03 -> 8.08,
    // K = 160 10.1 -> 9.8, K = 256 28.4 -> 26.1, x 100, K = 256 17.2 -> 18.6; 100,000 x 32, K = 160 18.3 -> 29.7.
    const bool use_wg = KP > 32 && join_wg_on() && launch_fits(grid_for_dies((size_t)N), 256) &&
                        D * (K - 24) > (MW == 2 ? 8000 : MW == 3 ? 6500 : MW == 4 ? 3000 : 95000);
    const unsigned short_groups = grid_for_dies(((size_t)N * (size_t)MW + kWaves - 1) / kWaves);
    const bool use_short = !use_wg && !w->bounds && ksteps <= 8 && launch_fits(short_groups, 64 * kWaves);
    // (the records of the reversed graph's builder are done with: the words take the place of the last ones, and are sorted from there)
    uint32_t* marks = use_short && w->staged && MW == 1 ? reinterpret_cast<uint32_t*>(w->bin_eq2) : nullptr;
    hipLaunchKernelGGL(k_join_bars, dim3((unsigned)((N + 255) / 256) + 1), dim3(256), 0, stream, jc, jc.scale(), knn_dist, N, K,
                       one_minus_gamma, w->bars, w->pass, marks ? 0 : (size_t)N * (size_t)K * (size_t)MW, knn_idx, old_idx);
    RSFK_HIP(hipGetLastError());
    // (the other forms read bars, not their codes)
    if (launch_rev(w, old_idx, N, K, stream, w->rev_bars && use_short)) return 1;
    if (use_wg) {
        const size_t lds_wg = (size_t)(kJwP + KP) * kJwRowBytes + (size_t)KP * 12 + (size_t)kJwP * 24;
#define RSFK_JOIN_WG(BV, NV)                                                                                                    \
        do {                                                                                                               \
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_explore_join_wg<BV, NV>),                         \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_wg));                       \
            hipLaunchKernelGGL((k_explore_join_wg<BV, NV>), dim3(grid_for_dies((size_t)N), parts), dim3(256), lds_wg, stream, jc, N, K,  \
                               old_idx, w->bars, w->offs, w->rev, w->pass, w->bounds, KP, join_pitch(D), ksteps, kappa,  \
                               any_rel, any_abs, w->div_m, w->div_s, order);                                                \
        } while (0)
        if (w->bounds && KP <= 128) RSFK_JOIN_WG(true, 3);
        else if (w->bounds) RSFK_JOIN_WG(true, 6);
        else if (KP <= 128) RSFK_JOIN_WG(false, 3);
        else RSFK_JOIN_WG(false, 6);
#undef RSFK_JOIN_WG
    } else if (use_short) {
        const dim3 grid(short_groups, parts), block(64 * kWaves);
#define RSFK_JOIN_SHORT(KSV, MANYV)                                                                                         \
        hipLaunchKernelGGL((k_explore_join_short<kWaves, KSV, MANYV>), grid, block, 0, stream, jc, N, K, old_idx, w->bars, w->offs, \
                           w->rev, w->rev_bars, w->pass, marks, MW, join_pitch(D), ksteps, kappa, any_rel, any_abs, w->div_m, w->div_s, order)
        if (MW == 1 && ksteps <= 2) RSFK_JOIN_SHORT(2, false);
        else if (MW == 1 && ksteps <= 4) RSFK_JOIN_SHORT(4, false);
        else if (MW == 1) RSFK_JOIN_SHORT(8, false);
        else if (ksteps <= 2) RSFK_JOIN_SHORT(2, true);
        else if (ksteps <= 4) RSFK_JOIN_SHORT(4, true);
        else RSFK_JOIN_SHORT(8, true);
#undef RSFK_JOIN_SHORT
        if (marks) {
            const size_t total = (size_t)N * (size_t)K;
            const int n_win = mark_windows(total), per = 1 << (kMarkWindow - kMarkPiece);
            const unsigned pieces = (unsigned)(((total - 1) >> kMarkPiece) + 1);
            int *by_window = w->sub_off, *by_piece = by_window + 32 * (size_t)n_win;
            hipLaunchKernelGGL(k_mark_clear, dim3((unsigned)((mark_ints(total) + 255) / 256)), dim3(256), 0, stream, by_window, (int)mark_ints(total));
            auto *to_windows = k_mark_scatter<true>, *to_pieces = k_mark_scatter<false>;
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(to_windows), hipFuncAttributeMaxDynamicSharedMemorySize, (int)mark_lds_bytes(n_win)));
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(to_pieces), hipFuncAttributeMaxDynamicSharedMemorySize, (int)mark_lds_bytes(per)));
            // (two workgroups fit a compute unit)
            const size_t tiles = (total + kMarkTile - 1) / kMarkTile;
            hipLaunchKernelGGL(to_windows, dim3((unsigned)std::min<size_t>(tiles, 512)), dim3(kMarkThreads), mark_lds_bytes(n_win), stream,
                               w->rev, marks, (const int2*)nullptr, w->offs + N, n_win, 32, by_window, w->bin_eq);
            hipLaunchKernelGGL(to_pieces, dim3((unsigned)(1024 / n_win + 1), (unsigned)n_win), dim3(kMarkThreads), mark_lds_bytes(per), stream,
                               (const int*)nullptr, (const uint32_t*)nullptr, w->bin_eq, by_window, per, 1, by_piece, w->bin_eq2);
            RSFK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k_mark_place), hipFuncAttributeMaxDynamicSharedMemorySize, 4 << kMarkPiece));
            hipLaunchKernelGGL(k_mark_place, dim3(pieces), dim3(kMarkThreads), 4 << kMarkPiece, stream, w->bin_eq2, by_piece, total, w->pass);
        }
    } else {
        auto* join = w->bounds ? (lines ? k_explore_join<kWaves, true, true> : k_explore_join<kWaves, true, false>)
                               : (lines ? k_explore_join<kWaves, false, true> : k_explore_join<kWaves, false, false>);
        hipLaunchKernelGGL(join, dim3(grid_for_dies(((size_t)N + kWaves - 1) / kWaves), parts), dim3(64 * kWaves), lds, stream, jc, N, K, old_idx,
                           w->bars, w->offs, w->rev, w->pass, w->bounds, KP, join_pitch(D), ksteps, kappa, any_rel, any_abs, wave_ints,
                           w->div_m, w->div_s, order);
    }
    RSFK_HIP(hipGetLastError());
    return 0;
}

}  // namespace rsfk
