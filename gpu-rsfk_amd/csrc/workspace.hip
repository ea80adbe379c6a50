// Device memory for the working buffers of a call (permutations, screening copies, exploration workspace).
//
// hipMalloc / hipFree of a few hundred megabytes cost tens to hundreds of microseconds each and a call needs
// about thirty of them, so blocks are kept after use and handed out again to the next call that asks for the
// same size on the same device (a build repeated with the same shapes allocates nothing).  A block that comes back when
// the cap is reached pushes out the blocks that have been idle longest (turned away itself, every later call of other shapes
// would allocate and free again: 2 GB for the pairs of a forest's buckets, 344,253 x 22, 15 trees 6.2 -> 40 ms a call after
// calls that had filled the cap).  Idle blocks are
// capped at RSFK_WORKSPACE_POOL_MB megabytes (default: a quarter of the device memory, at most 16 GiB; 0 keeps
// nothing); rsfk_release_workspace() returns all of them to the driver.
// The reference allocates and frees inside every tree level (src/rsfk.cu:640-1180).
#include "rsfk_common.hpp"
#include <algorithm>
#include <cstdlib>
#include <map>
#include <cstring>
#include <mutex>
#include <vector>

namespace rsfk {

namespace {

struct Pool {
    std::mutex mu;
    struct Idle {
        void* p;
        unsigned long long since;
    };
    std::multimap<std::pair<int, size_t>, Idle> idle;      // (device, bytes) -> block
    unsigned long long frees = 0;
    std::map<void*, std::pair<int, size_t>> live;           // blocks handed out
    size_t idle_bytes = 0;
    size_t idle_cap = 0;                                    // set on first use
    bool cap_known = false;
};

// most idle bytes the pool keeps (asked of the device once)
size_t idle_cap_locked(Pool& P)
{
    if (!P.cap_known) {
        P.cap_known = true;
        size_t free_b = 0, total_b = 0;
        P.idle_cap = (size_t)4 << 30;
        if (hipMemGetInfo(&free_b, &total_b) == hipSuccess) P.idle_cap = std::min<size_t>(total_b / 4, (size_t)16 << 30);
        const char* e = std::getenv("RSFK_WORKSPACE_POOL_MB");
        if (e && *e) P.idle_cap = (size_t)std::max(0ll, std::atoll(e)) << 20;
    }
    return P.idle_cap;
}

Pool& pool()
{
    static Pool p;
    return p;
}

}  // namespace

namespace {
// must: a block the caller cannot do without (idle blocks are given back to make room, the error text is set);
// otherwise one plain attempt that leaves the pool and the error text alone
int ws_alloc_impl(void** out, size_t bytes, bool must)
{
    *out = nullptr;
    if (bytes == 0) bytes = 1;
    bytes = (bytes + 255) & ~(size_t)255;
    int dev = 0;
    RSFK_HIP(hipGetDevice(&dev));
    Pool& P = pool();
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.idle.find({dev, bytes});
        if (it != P.idle.end()) {
            *out = it->second.p;
            P.idle.erase(it);
            P.idle_bytes -= bytes;
            P.live[*out] = {dev, bytes};
            return 0;
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess && !must) {
        (void)hipGetLastError();
        return 1;
    }
    if (e != hipSuccess) {
        // give the idle blocks back and try once more
        (void)hipGetLastError();
        ws_release_all();
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        set_last_error(std::string("out of device memory (") + std::to_string(bytes) + " bytes): " + hipGetErrorString(e));
        (void)hipDeviceSynchronize();       // (the caller's guards hand their blocks back on the way out)
        return 1;
    }
    std::lock_guard<std::mutex> lock(P.mu);
    P.live[p] = {dev, bytes};
    *out = p;
    return 0;
}
}  // namespace

int ws_alloc(void** out, size_t bytes) { return ws_alloc_impl(out, bytes, true); }

// A block the caller can do without (it only makes something faster): nonzero, with nothing else changed, when the
// device does not have the room, or when it has RSFK_OPTIONAL_MB megabytes or more (read at every call: tests change it).
int ws_try_alloc(void** out, size_t bytes)
{
    *out = nullptr;
    const char* most = std::getenv("RSFK_OPTIONAL_MB");
    if (most && *most && (long long)(bytes >> 20) >= std::atoll(most)) return 1;
    return ws_alloc_impl(out, bytes, false);
}

// The caller has made sure that no work that uses the block is still running.
void ws_free(void* p)
{
    if (!p) return;
    Pool& P = pool();
    std::vector<void*> out;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.live.find(p);
        if (it == P.live.end()) {           // not ours
            out.push_back(p);
        } else {
            const std::pair<int, size_t> key = it->second;
            const size_t cap = idle_cap_locked(P);
            P.live.erase(it);
            if (key.second > cap) {
                out.push_back(p);
            } else {
                while (P.idle_bytes + key.second > cap) {
                    auto oldest = P.idle.begin();
                    for (auto i = P.idle.begin(); i != P.idle.end(); ++i)
                        if (i->second.since < oldest->second.since) oldest = i;
                    P.idle_bytes -= oldest->first.second;
                    out.push_back(oldest->second.p);
                    P.idle.erase(oldest);
                }
                P.idle.insert({key, {p, P.frees++}});
                P.idle_bytes += key.second;
            }
        }
    }
    for (void* q : out) (void)hipFree(q);
}

// ---- pinned host memory and side streams --------------------------------------------------------------------------
//
// A call needs a few pinned blocks (counters that come back from the device, small arrays on their way) and most calls
// a second stream.  hipHostMalloc + hipHostFree take 26 us and hipStreamCreate + Destroy 57 us, which
// together was a fifth of a small call (10,000 x 32 points, 4 trees: 0.35 of 1.8 ms), so both are kept for the next
// call: at most 64 MB of idle pinned blocks (rounded up to powers of two) and eight idle streams.
namespace {

struct HostPool {
    std::mutex mu;
    std::multimap<std::pair<int, size_t>, void*> idle;     // (device, bytes) -> block
    std::map<void*, std::pair<int, size_t>> live;
    size_t idle_bytes = 0;
    std::vector<std::pair<int, hipStream_t>> streams;       // idle ones and their devices
};
constexpr size_t kPinIdleMax = (size_t)64 << 20;
constexpr size_t kStreamsIdleMax = 8;

HostPool& host_pool()
{
    static HostPool p;
    return p;
}

}  // namespace

int pin_alloc(void** out, size_t bytes)
{
    *out = nullptr;
    size_t b = 4096;
    while (b < bytes) b <<= 1;
    int dev = 0;
    RSFK_HIP(hipGetDevice(&dev));
    HostPool& P = host_pool();
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.idle.find({dev, b});
        if (it != P.idle.end()) {
            *out = it->second;
            P.idle.erase(it);
            P.idle_bytes -= b;
            P.live[*out] = {dev, b};
            return 0;
        }
    }
    void* p = nullptr;
    RSFK_HIP(hipHostMalloc(&p, b));
    std::lock_guard<std::mutex> lock(P.mu);
    P.live[p] = {dev, b};
    *out = p;
    return 0;
}

// The caller has made sure that no copy or kernel that uses the block is still running.
void pin_free(void* p)
{
    if (!p) return;
    HostPool& P = host_pool();
    {
        std::lock_guard<std::mutex> lock(P.mu);
        auto it = P.live.find(p);
        if (it != P.live.end()) {
            const std::pair<int, size_t> key = it->second;
            P.live.erase(it);
            if (P.idle_bytes + key.second <= kPinIdleMax) {
                P.idle.insert({key, p});
                P.idle_bytes += key.second;
                return;
            }
        }
    }
    (void)hipHostFree(p);
}

// A non-blocking stream of default priority on the current device.
int stream_take(hipStream_t* out)
{
    *out = nullptr;
    int dev = 0;
    RSFK_HIP(hipGetDevice(&dev));
    HostPool& P = host_pool();
    {
        std::lock_guard<std::mutex> lock(P.mu);
        for (size_t i = 0; i < P.streams.size(); ++i)
            if (P.streams[i].first == dev) {
                *out = P.streams[i].second;
                P.streams.erase(P.streams.begin() + (ptrdiff_t)i);
                return 0;
            }
    }
    RSFK_HIP(hipStreamCreateWithFlags(out, hipStreamNonBlocking));
    return 0;
}

// Everything queued on the stream has been waited for.
void stream_give(hipStream_t s)
{
    if (!s) return;
    int dev = 0;
    HostPool& P = host_pool();
    if (hipGetDevice(&dev) == hipSuccess) {
        std::lock_guard<std::mutex> lock(P.mu);
        if (P.streams.size() < kStreamsIdleMax) {
            P.streams.push_back({dev, s});
            return;
        }
    }
    (void)hipStreamDestroy(s);
}

// Polling pinned memory takes 6 us from the launch of the kernel that writes it, a copy and a synchronisation 14.  When
// the word does not come for a while the stream is asked how it is: an error, or a stream that has finished without
// writing the word, ends the wait.
int wait_for_word(const int* word, int want, hipStream_t stream)
{
    const auto seen = [&] { return __atomic_load_n(word, __ATOMIC_ACQUIRE) == want; };
    for (long long spin = 1; !seen(); ++spin) {
        if ((spin & 0xffff) != 0) continue;
        const hipError_t e = hipStreamQuery(stream);
        if (e == hipErrorNotReady) continue;
        (void)hipGetLastError();
        RSFK_HIP(hipStreamSynchronize(stream));
        RSFK_CHECK(seen(), "a kernel has ended without its answer");
    }
    return 0;
}

namespace {
struct Fetched {
    int word[kFetchMost];
    int seq;
};
__global__ void k_fetch(const int* __restrict__ a, int na, const int* __restrict__ b, int nb, Fetched* out)
{
    for (int i = 0; i < na; ++i) out->word[i] = a[i];
    for (int i = 0; i < nb; ++i) out->word[na + i] = b[i];
    __hip_atomic_store(&out->seq, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__global__ void k_fetch_total(const int* __restrict__ a, int n, int pitch, Fetched* out)
{
    int v = (int)threadIdx.x < n ? a[(size_t)threadIdx.x * (size_t)pitch] : 0;
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if (threadIdx.x != 0) return;
    out->word[0] = v;
    __hip_atomic_store(&out->seq, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// One workgroup of 256 threads.
__global__ void k_fetch_total64(const unsigned long long* __restrict__ a, int n, int pitch, Fetched* out)
{
    __shared__ unsigned long long part[256];
    unsigned long long t = 0;
    for (int i = threadIdx.x; i < n; i += 256) t += a[(size_t)i * (size_t)pitch];
    part[threadIdx.x] = t;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    out->word[0] = (int)(unsigned)part[0];
    out->word[1] = (int)(unsigned)(part[0] >> 32);
    __hip_atomic_store(&out->seq, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
// One workgroup of 256 threads.
__global__ void k_fetch_sum(const float* __restrict__ a, int n, Fetched* out)
{
    __shared__ float part[256];
    float t = 0.0f;
    for (int i = threadIdx.x; i < n; i += 256) t += a[i];
    part[threadIdx.x] = t;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    out->word[0] = __float_as_int(part[0]);
    __hip_atomic_store(&out->seq, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
}  // namespace

int fetch_words(const int* a, int na, const int* b, int nb, int* host, hipStream_t stream)
{
    const int n = na + nb;
    RSFK_CHECK(n >= 1 && n <= kFetchMost, "fetch: too many words");
    void* p = nullptr;
    if (pin_alloc(&p, sizeof(Fetched))) return 1;
    Fetched* f = static_cast<Fetched*>(p);
    __atomic_store_n(&f->seq, 0, __ATOMIC_RELEASE);
    hipLaunchKernelGGL(k_fetch, dim3(1), dim3(1), 0, stream, a, na, b, nb, f);
    const hipError_t e = hipGetLastError();
    const int rc = e != hipSuccess ? 1 : wait_for_word(&f->seq, 1, stream);
    if (e != hipSuccess) set_last_error(std::string("fetch: ") + hipGetErrorString(e));
    for (int i = 0; i < n && !rc; ++i) host[i] = f->word[i];
    pin_free(p);
    return rc;
}

int fetch_total(const int* a, int n, int pitch, int* host, hipStream_t stream)
{
    RSFK_CHECK(n >= 1 && n <= 64, "fetch: too many words");
    void* p = nullptr;
    if (pin_alloc(&p, sizeof(Fetched))) return 1;
    Fetched* f = static_cast<Fetched*>(p);
    __atomic_store_n(&f->seq, 0, __ATOMIC_RELEASE);
    hipLaunchKernelGGL(k_fetch_total, dim3(1), dim3(64), 0, stream, a, n, pitch, f);
    const hipError_t e = hipGetLastError();
    const int rc = e != hipSuccess ? 1 : wait_for_word(&f->seq, 1, stream);
    if (e != hipSuccess) set_last_error(std::string("fetch: ") + hipGetErrorString(e));
    if (!rc) *host = f->word[0];
    pin_free(p);
    return rc;
}

int fetch_total(const unsigned long long* a, int n, int pitch, unsigned long long* host, hipStream_t stream)
{
    void* p = nullptr;
    if (pin_alloc(&p, sizeof(Fetched))) return 1;
    Fetched* f = static_cast<Fetched*>(p);
    __atomic_store_n(&f->seq, 0, __ATOMIC_RELEASE);
    hipLaunchKernelGGL(k_fetch_total64, dim3(1), dim3(256), 0, stream, a, n, pitch, f);
    const hipError_t e = hipGetLastError();
    const int rc = e != hipSuccess ? 1 : wait_for_word(&f->seq, 1, stream);
    if (e != hipSuccess) set_last_error(std::string("fetch: ") + hipGetErrorString(e));
    if (!rc) *host = (unsigned)f->word[0] | (unsigned long long)(unsigned)f->word[1] << 32;
    pin_free(p);
    return rc;
}

int fetch_sum(const float* a, int n, float* host, hipStream_t stream)
{
    void* p = nullptr;
    if (pin_alloc(&p, sizeof(Fetched))) return 1;
    Fetched* f = static_cast<Fetched*>(p);
    __atomic_store_n(&f->seq, 0, __ATOMIC_RELEASE);
    hipLaunchKernelGGL(k_fetch_sum, dim3(1), dim3(256), 0, stream, a, n, f);
    const hipError_t e = hipGetLastError();
    const int rc = e != hipSuccess ? 1 : wait_for_word(&f->seq, 1, stream);
    if (e != hipSuccess) set_last_error(std::string("fetch: ") + hipGetErrorString(e));
    if (!rc) std::memcpy(host, &f->word[0], sizeof(float));
    pin_free(p);
    return rc;
}

void host_pool_release()
{
    HostPool& P = host_pool();
    std::vector<void*> blocks;
    std::vector<std::pair<int, hipStream_t>> streams;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        for (auto& kv : P.idle) blocks.push_back(kv.second);
        P.idle.clear();
        P.idle_bytes = 0;
        streams.swap(P.streams);
    }
    for (void* b : blocks) (void)hipHostFree(b);
    for (auto& s : streams) (void)hipStreamDestroy(s.second);
}

void ws_release_all()
{
    Pool& P = pool();
    std::vector<void*> blocks;
    {
        std::lock_guard<std::mutex> lock(P.mu);
        for (auto& kv : P.idle) blocks.push_back(kv.second.p);
        P.idle.clear();
        P.idle_bytes = 0;
    }
    for (void* b : blocks) (void)hipFree(b);
}

}  // namespace rsfk
