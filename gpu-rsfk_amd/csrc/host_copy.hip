// Copies between pageable host arrays (what a ctypes caller hands over: numpy buffers) and device memory.
//
// hipMemcpy on pageable memory moves the bytes through a bounce buffer on one thread, and its time has little to do
// with the size of a small array (320 KB to the device: 133 us, 14 us from pinned memory).  So:
//   small arrays (all arrays of a call together below 4 MB) go through one pinned block on the calling thread, in
//     pieces, the memcpy of a piece beside the DMA of the piece before; copies to the device are only queued on the
//     caller's stream (2.4 MB: 101 us with hipMemcpy, 56 us here).
//   large ones: host threads take pieces of 2 MB in turn, each through its own pair of pinned buffers (hipHostMalloc;
//     registering the caller's memory is not an option) on one of two streams: the memcpy of one piece overlaps the DMA of
//     the previous one and the threads overlap each other.  What bounds it is the link (57 GB/s each way); one thread
//     copies 10 GB/s or so, less where the destination's pages are touched for the first time, hence eight threads.
//     Four threads with pieces of 8 MB, the form before, had nothing to overlap below 64 MB.
//   results of large calls (HostResult): the pages of a fresh array do not exist yet, and making them takes more than the copy
//     (44 MB: 2.7 ms into fresh pages, 1.2 into present ones), so a thread makes them while the device works
//     (123,457 x 37, K = 45, 12 trees, one pass: 6.65 -> 6.41 ms for the call).  Small results
//     come and go with the heap's own pages (and a thread is 13 us).  (Letting such threads take part in the copy as well, with
//     pieces of 256 KB: 5 MB 256 -> 370 us, 44 MB 1.16 -> 1.28 ms; the calls per piece cost more than starting threads.)
// The buffers and streams are kept for the next call; rsfk_release_workspace() frees them.
#include "rsfk_common.hpp"
#include "forest.hpp"
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>
#include <sys/mman.h>
#include <unistd.h>

namespace rsfk {

namespace {

constexpr int kCopyThreads = 8;
constexpr int kCopyStreams = 2;
constexpr size_t kPiece = (size_t)2 << 20;          // bytes per pinned buffer of a thread
constexpr size_t kSmall = (size_t)4 << 20;          // up to here on the calling thread
constexpr size_t kSmallPiece = (size_t)512 << 10;

struct Lane {
    void* pinned[2] = {nullptr, nullptr};
    hipEvent_t done[2] = {nullptr, nullptr};
};

struct Lanes {
    std::mutex mu;
    int device = -1;
    Lane lane[kCopyThreads];
    hipStream_t stream[kCopyStreams] = {};
    bool ready = false;
};

Lanes& lanes()
{
    static Lanes l;
    return l;
}

void free_lanes_locked(Lanes& L)
{
    for (Lane& a : L.lane) {
        for (int i = 0; i < 2; ++i) {
            if (a.pinned[i]) (void)hipHostFree(a.pinned[i]);
            if (a.done[i]) (void)hipEventDestroy(a.done[i]);
            a.pinned[i] = nullptr;
            a.done[i] = nullptr;
        }
    }
    for (hipStream_t& s : L.stream) {
        if (s) (void)hipStreamDestroy(s);
        s = nullptr;
    }
    L.ready = false;
    L.device = -1;
}

int make_lanes_locked(Lanes& L, int dev)
{
    if (L.ready && L.device == dev) return 0;
    free_lanes_locked(L);
    for (Lane& a : L.lane) {
        for (int i = 0; i < 2; ++i) {
            RSFK_HIP(hipHostMalloc(&a.pinned[i], kPiece));
            RSFK_HIP(hipEventCreateWithFlags(&a.done[i], hipEventDisableTiming));
        }
    }
    for (hipStream_t& s : L.stream) RSFK_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    L.device = dev;
    L.ready = true;
    return 0;
}

struct Piece {
    char* dev;
    char* host;
    size_t bytes;
};

// one thread: pieces in turn until none is left
void run_lane(Lane& a, hipStream_t stream, int dev, const std::vector<Piece>& pieces, std::atomic<size_t>& next, bool to_device, std::atomic<int>& err)
{
    if (hipSetDevice(dev) != hipSuccess) { err = 1; return; }
    Piece in[2] = {};
    int n = 0;
    auto finish = [&](int b) {
        if (hipEventSynchronize(a.done[b]) != hipSuccess) { err = 1; return; }
        if (!to_device) std::memcpy(in[b].host, a.pinned[b], in[b].bytes);
    };
    for (; !err; ++n) {
        const size_t i = next.fetch_add(1);
        if (i >= pieces.size()) break;
        const int b = n & 1;
        if (n >= 2) finish(b);                       // the piece that used this buffer two steps ago
        if (err) break;
        in[b] = pieces[i];
        if (to_device) std::memcpy(a.pinned[b], in[b].host, in[b].bytes);
        const hipError_t e = to_device ? hipMemcpyAsync(in[b].dev, a.pinned[b], in[b].bytes, hipMemcpyHostToDevice, stream)
                                       : hipMemcpyAsync(a.pinned[b], in[b].dev, in[b].bytes, hipMemcpyDeviceToHost, stream);
        if (e != hipSuccess || hipEventRecord(a.done[b], stream) != hipSuccess) { err = 1; return; }
    }
    for (int k = std::max(0, n - 2); k < n && !err; ++k) finish(k & 1);
}

int large_copy(const std::vector<Piece>& pieces, bool to_device)
{
    int dev = 0;
    RSFK_HIP(hipGetDevice(&dev));
    Lanes& L = lanes();
    std::lock_guard<std::mutex> lock(L.mu);            // one such copy at a time
    if (make_lanes_locked(L, dev)) return 1;
    std::atomic<int> err{0};
    std::atomic<size_t> next{0};
    const int n_threads = (int)std::min<size_t>(kCopyThreads, pieces.size());
    std::vector<std::thread> th;
    th.reserve(kCopyThreads);
    try {
        for (int t = 1; t < n_threads; ++t)
            th.emplace_back(run_lane, std::ref(L.lane[t]), L.stream[t % kCopyStreams], dev, std::cref(pieces), std::ref(next), to_device, std::ref(err));
    } catch (const std::system_error&) {
        // (a process at its limit of threads: those that are there take the pieces in turn)
    }
    run_lane(L.lane[0], L.stream[0], dev, pieces, next, to_device, err);
    for (auto& t : th) t.join();
    RSFK_CHECK(err == 0, "copy between host and device failed");
    return 0;
}

std::vector<Piece> cut(const HostArray* a, int n, size_t piece)
{
    std::vector<Piece> out;
    for (int i = 0; i < n; ++i)
        for (size_t at = 0; at < a[i].bytes; at += piece)
            out.push_back({static_cast<char*>(a[i].dev) + at, static_cast<char*>(a[i].host) + at, std::min(piece, a[i].bytes - at)});
    return out;
}

size_t total_bytes(const HostArray* a, int n)
{
    size_t t = 0;
    for (int i = 0; i < n; ++i) t += a[i].bytes;
    return t;
}

}  // namespace

HostStage::~HostStage()
{
    if (block_) {
        (void)hipStreamSynchronize(stream_);           // (only on an error path is anything still queued)
        pin_free(block_);
    }
}

int HostStage::to_device(const HostArray* a, int n, hipStream_t stream)
{
    const size_t total = total_bytes(a, n);
    if (total == 0) return 0;
    if (total > kSmall || block_) return large_copy(cut(a, n, kPiece), true);
    if (pin_alloc(&block_, total)) return 1;
    stream_ = stream;
    char* at = static_cast<char*>(block_);
    for (const Piece& p : cut(a, n, kSmallPiece)) {
        std::memcpy(at, p.host, p.bytes);
        RSFK_HIP(hipMemcpyAsync(p.dev, at, p.bytes, hipMemcpyHostToDevice, stream));
        at += p.bytes;
    }
    return 0;
}

int copy_to_host(const HostArray* a, int n, hipStream_t stream)
{
    const size_t total = total_bytes(a, n);
    if (total == 0) return 0;
    if (total > kSmall) {
        RSFK_HIP(hipStreamSynchronize(stream));        // the copies run on streams of their own
        return large_copy(cut(a, n, kPiece), false);
    }
    struct Guard {
        void* p = nullptr;
        ~Guard() { pin_free(p); }
    } block;
    if (pin_alloc(&block.p, total)) return 1;
    const std::vector<Piece> pieces = cut(a, n, 2 * kSmallPiece);
    char* at = static_cast<char*>(block.p);
    for (const Piece& p : pieces) {
        RSFK_HIP(hipMemcpyAsync(at, p.dev, p.bytes, hipMemcpyDeviceToHost, stream));
        at += p.bytes;
    }
    RSFK_HIP(hipStreamSynchronize(stream));
    at = static_cast<char*>(block.p);
    for (const Piece& p : pieces) {
        std::memcpy(p.host, at, p.bytes);
        at += p.bytes;
    }
    return 0;
}

#ifndef MADV_POPULATE_WRITE
#define MADV_POPULATE_WRITE 23
#endif

void HostResult::begin(const HostArray* a, int n)
{
    if (total_bytes(a, n) <= kSmall || pages_.joinable()) return;
    try {
        const std::vector<Piece> pieces = cut(a, n, (size_t)4 << 20);
        pages_ = std::thread([this, pieces] {
            const uintptr_t page = (uintptr_t)sysconf(_SC_PAGESIZE);
            for (const Piece& p : pieces) {
                if (stop_.load(std::memory_order_relaxed)) break;
                // the pages a piece lies on hold bytes of the array, so they are there to be written; nothing in them changes
                const uintptr_t first = reinterpret_cast<uintptr_t>(p.host) / page * page;
                const uintptr_t end = (reinterpret_cast<uintptr_t>(p.host) + p.bytes + page - 1) / page * page;
                if (madvise(reinterpret_cast<void*>(first), end - first, MADV_POPULATE_WRITE) != 0) break;      // (an old kernel: the copy makes them)
            }
        });
    } catch (const std::exception&) {
        // no memory, or no thread: the copy makes the pages
    }
}

HostResult::~HostResult()
{
    stop_ = true;
    if (pages_.joinable()) pages_.join();
}

int HostResult::finish(const HostArray* a, int n, hipStream_t stream)
{
    stop_ = true;                                        // (what is left is made faster by the eight threads of the copy)
    if (pages_.joinable()) pages_.join();
    return copy_to_host(a, n, stream);
}

void release_copy_buffers()
{
    Lanes& L = lanes();
    std::lock_guard<std::mutex> lock(L.mu);
    free_lanes_locked(L);
}

}  // namespace rsfk
