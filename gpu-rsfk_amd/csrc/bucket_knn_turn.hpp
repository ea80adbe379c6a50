// A turn of K-NN rows: up to 64 candidates of several rows, one per lane, go into their rows together, by one wavefront
// (bucket_knn_rows_screen.hip, bucket_knn_screen.hip).  The rows pass through LDS as keys; every lane counts the entries of its row
// below its candidate, sees whether the row holds the candidate already, and counts the row's other new candidates below it: that is
// the candidate's slot, and an entry of the row moves up by the candidates that end below it.  Nothing is inserted one by one.
#pragma once
#include "rsfk_common.hpp"
#include "knn_list.hpp"

namespace rsfk {

constexpr int kTurnFlight = 4;                // rows of kTurnFlight * 64 slots together at a time
constexpr int kTurnRoom = 272;                // ... and their room in LDS, in slots
constexpr int kTurnMostRows = 16;
constexpr int kTurnGap = 3;
static_assert(64 + kTurnGap * kTurnMostRows <= 128, "the places of a turn's candidates");

// Per wavefront; slot[r].x (the point of row r) is the caller's, the other words of a slot are zero when the turn begins.
struct TurnLds {
    double row[kTurnRoom];                    // K-NN rows, as keys
    float cand[128];                          // the distances of new candidates, kTurnGap free places (+inf) after every row's
    int4 slot[kTurnMostRows];                 // per row: its point, -, the final places of new candidates (two words)
};

inline int turn_per_k(int K) { return (65536 + K - 1) / K; }

struct RowTurn {
    int K, row_pitch, n_room;                 // n_room: rows of a turn at most
    int rk[kTurnFlight];                      // row << 8 | entry of this lane's slots of the buffer: slot q is entry q % K of row q / K
    int xi[kTurnFlight], xd[kTurnFlight];

    // per_k = turn_per_k(K): q / K = (q * per_k) >> 16 for q < 256, K <= 64
    __device__ __forceinline__ RowTurn(int K_, int per_k) : K(K_)
    {
        row_pitch = (K + 3) & ~1;                                 // (16 bytes from row to row on top: they start in different banks)
        n_room = min(kTurnMostRows, min((64 * kTurnFlight * per_k) >> 16, kTurnRoom / row_pitch));
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x) {
            const int q = lane_id() + 64 * x, r = (q * per_k) >> 16;
            rk[x] = r << 8 | (q - r * K);
        }
    }

    // the rows of slot[0 .. n_rows) on their way
    __device__ __forceinline__ void request(const TurnLds& L, int n_rows, const int* __restrict__ knn_idx,
                                            const float* __restrict__ knn_dist)
    {
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x) {
            xi[x] = -1;
            xd[x] = 0;
            if ((rk[x] >> 8) < n_rows) {
                const size_t at = (size_t)L.slot[rk[x] >> 8].x * (size_t)K + (rk[x] & 255);
                xi[x] = knn_idx[at];
                xd[x] = __float_as_int(knn_dist[at]);
            }
        }
    }

    // enter: this lane has a candidate, point cid at distance d (not above the last slot of its row), for row prow; the candidates of
    // that row are those of lanes lo .. lo + count - 1 (of the n lanes with candidates, in the order of the rows).
    __device__ __forceinline__ void merge(TurnLds& L, int n_rows, int n, bool enter, int prow, int lo, int count, int cid, float d,
                                          int* __restrict__ knn_idx, float* __restrict__ knn_dist)
    {
        const int lane = lane_id();
        const double key = pair_key(d, cid);
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x) {
            asm("" : "+v"(xi[x]), "+v"(xd[x]));                   // (or the keys are computed where the loads are, which then wait for each other)
        }
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x)
            if ((rk[x] >> 8) < n_rows) L.row[(rk[x] >> 8) * row_pitch + (rk[x] & 255)] = pair_key(__int_as_float(xd[x]), xi[x]);
        wave_lds_sync();
        // against the row: is the candidate there already, how many entries are below it
        int below = 0;
        bool there = false, level;
        {
            const double* r = L.row + (enter ? prow * row_pitch : 0);
#pragma unroll 4
            for (int k = 0; k < K / 2; ++k) {
                const double2 v = *reinterpret_cast<const double2*>(r + 2 * k);
                there |= __double2loint(v.x) == cid || __double2loint(v.y) == cid;
                below += v.x < key ? 1 : 0;
                below += v.y < key ? 1 : 0;
            }
            if (K & 1) {
                const double v = r[K - 1];
                there |= __double2loint(v) == cid;
                below += v < key ? 1 : 0;
            }
            level = __double2hiint(r[max(below - 1, 0)]) == __double2hiint(key) ||
                    __double2hiint(r[min(below, K - 1)]) == __double2hiint(key);
        }
        // against the member's other new candidates: by distance alone, where that decides
        const bool fresh = enter && !there;
        const int end = fresh ? min(count, n - lo) : 0;
        const int mine_at = kTurnGap * prow + lo;
        *reinterpret_cast<float2*>(&L.cand[2 * lane]) = make_float2(INFINITY, INFINITY);
        wave_lds_sync();
        if (fresh) L.cand[kTurnGap * prow + lane] = d;
        wave_lds_sync();
        const int below_row = below;
        for (int k = 0; ballot64(k < end) != 0; k += 4) {
            const float* c = L.cand + (k < end ? mine_at + k : 124);
#pragma unroll
            for (int u = 0; u < 4; ++u) below += c[u] < d ? 1 : 0;
        }
        bool in = fresh && below < K;
        uint32_t* places = reinterpret_cast<uint32_t*>(&L.slot[prow]) + 2;
        const uint32_t bit = 1u << (below & 31);
        const bool taken = in && (atomicOr(places + (below >> 5), bit) & bit) != 0;
        if (ballot64(taken || (fresh && level)) != 0) {
            // (two candidates at one distance, with or without an entry of the row between them: the indices decide)
            if (in) atomicAnd(places + (below >> 5), ~bit);
            below = below_row;
            for (int k = 0; k < n; ++k) {
                const bool other = read_lane_i(fresh ? prow : -1, k) == prow;
                below += other && pair_above(d, cid, read_lane_f(d, k), read_lane_i(cid, k)) ? 1 : 0;
            }
            in = fresh && below < K;
            if (in) atomicOr(places + (below >> 5), 1u << (below & 31));
        }
        if (ballot64(in) == 0) return;
        wave_lds_sync();
        // the new rows: an entry moves up by the candidates that end below it
        double xv[kTurnFlight];
        uint32_t is_new = 0, changed = 0;
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x) {
            xv[x] = 0.0;
            if ((rk[x] >> 8) < n_rows) {
                const int k = rk[x] & 255;
                const int2 m2 = *(reinterpret_cast<const int2*>(&L.slot[rk[x] >> 8]) + 1);
                const uint64_t m = ((uint64_t)(uint32_t)m2.y << 32) | (uint32_t)m2.x;
                if (m != 0) changed |= 1u << x;
                if ((m >> k) & 1) is_new |= 1u << x;
                xv[x] = L.row[(rk[x] >> 8) * row_pitch + k - __popcll(m & ((1ull << k) - 1))];
            }
        }
        wave_lds_sync();
        if (in) L.row[prow * row_pitch + below] = key;
        wave_lds_sync();
#pragma unroll
        for (int x = 0; x < kTurnFlight; ++x) {
            if ((is_new >> x) & 1) xv[x] = L.row[(rk[x] >> 8) * row_pitch + (rk[x] & 255)];
            if ((changed >> x) & 1) {
                const size_t at = (size_t)L.slot[rk[x] >> 8].x * (size_t)K + (rk[x] & 255);
                knn_idx[at] = __double2loint(xv[x]);
                knn_dist[at] = pair_dist(xv[x]);
            }
        }
    }
};

}  // namespace rsfk
