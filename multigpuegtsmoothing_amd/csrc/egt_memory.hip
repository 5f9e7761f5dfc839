// Device memory cache for handle allocations.
//
// A handle allocates its point arrays, tables, rows and scratch once per stage and frees all of them when
// it is destroyed; a caller that smooths one cloud after another would otherwise pay hipMalloc and hipFree
// (each a device-wide synchronization) for every buffer of every cloud. Blocks released by a handle are
// kept per device and handed to later requests of a similar size. Release happens only after the device
// has drained (DBuf::free synchronizes first), so a cached block is never in use by in-flight work and can
// be handed to any stream. Cached bytes per device are capped (EGT_DEVICE_CACHE_MB, default 32768); a
// failed hipMalloc returns the device's cached blocks to the driver and tries once more.
// egt_release_cached_memory() returns every cached block.
//
// Beside them, up to IDLE_LANES stream and pinned block pairs per device: creating and destroying a stream takes
// 58 us, a tenth of a call on 1,500 points, and a copy into pinned memory 9 us less than one into pageable memory.
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include "egt_internal.h"

namespace egt {
namespace {

struct Cache {
    std::mutex mu;
    std::map<int, std::multimap<size_t, void*>> free_blocks;  // device -> (capacity, block)
    std::map<int, size_t> cached;                             // device -> cached bytes
    std::map<int, std::vector<Lane>> lanes;                   // device -> idle streams with their pinned blocks
};

Cache& cache() {
    static Cache* c = new Cache;  // never destroyed: HIP may already be torn down at static destruction
    return *c;
}

size_t cache_cap_bytes() {
    static size_t cap = [] {
        const char* e = std::getenv("EGT_DEVICE_CACHE_MB");
        const long long mb = e ? std::atoll(e) : 32768;
        return (size_t)(mb < 0 ? 0 : mb) << 20;
    }();
    return cap;
}

constexpr size_t GRAIN = 256;
constexpr size_t IDLE_LANES = 16;

void destroy_lane(const Lane& l) {
    if (l.stream) (void)hipStreamDestroy(l.stream);
    if (l.pinned) (void)hipHostFree(l.pinned);
}

// Frees the cached blocks of device dev (the caller holds the lock and has dev current).
size_t drop_device(Cache& c, int dev) {
    size_t freed = 0;
    auto& fb = c.free_blocks[dev];
    for (auto& kv : fb) {
        (void)hipFree(kv.second);
        freed += kv.first;
    }
    fb.clear();
    c.cached[dev] = 0;
    return freed;
}

}  // namespace

void* device_alloc(size_t bytes, size_t* capacity) {
    bytes = (std::max<size_t>(bytes, 1) + GRAIN - 1) / GRAIN * GRAIN;
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    Cache& c = cache();
    {
        std::lock_guard<std::mutex> lock(c.mu);
        auto& fb = c.free_blocks[dev];
        auto it = fb.lower_bound(bytes);
        // reuse the smallest cached block that fits, unless it would waste more than the request itself
        if (it != fb.end() && it->first <= 2 * bytes + (1u << 20)) {
            void* p = it->second;
            *capacity = it->first;
            c.cached[dev] -= it->first;
            fb.erase(it);
            return p;
        }
    }
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        {
            std::lock_guard<std::mutex> lock(c.mu);
            drop_device(c, dev);
        }
        e = hipMalloc(&p, bytes);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();
        throw HipError{e, "hipMalloc of " + std::to_string(bytes) + " bytes"};
    }
    *capacity = bytes;
    return p;
}

void device_release(void* p, size_t capacity) {
    if (!p) return;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)hipFree(p);
        return;
    }
    Cache& c = cache();
    std::lock_guard<std::mutex> lock(c.mu);
    if (c.cached[dev] + capacity > cache_cap_bytes()) {
        (void)hipFree(p);
        return;
    }
    c.free_blocks[dev].emplace(capacity, p);
    c.cached[dev] += capacity;
}

Lane lane_acquire() {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    Cache& c = cache();
    {
        std::lock_guard<std::mutex> lock(c.mu);
        std::vector<Lane>& idle = c.lanes[dev];
        if (!idle.empty()) {
            const Lane l = idle.back();
            idle.pop_back();
            return l;
        }
    }
    Lane l;
    l.device = dev;
    HIP_CHECK(hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking));
    if (hipHostMalloc(&l.pinned, PINNED_BYTES, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        l.pinned = nullptr;  // read-backs then go straight to the caller's memory
    }
    return l;
}

void lane_release(const Lane& l) {
    if (!l.stream) return;
    // a stream in capture or in error is not for another handle
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(l.stream, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone &&
        hipStreamQuery(l.stream) == hipSuccess) {
        Cache& c = cache();
        std::lock_guard<std::mutex> lock(c.mu);
        std::vector<Lane>& idle = c.lanes[l.device];
        if (idle.size() < IDLE_LANES) {
            idle.push_back(l);
            return;
        }
    }
    (void)hipGetLastError();
    destroy_lane(l);
}

void fetch(const Lane& l, std::initializer_list<HostCopy> copies) {
    auto step = [](const HostCopy& c) { return (c.bytes + 15) / 16 * 16; };
    auto fits = [&](size_t used, const HostCopy& c) { return l.pinned && used + c.bytes <= PINNED_BYTES; };
    char* const p = static_cast<char*>(l.pinned);
    size_t used = 0;
    for (const HostCopy& c : copies) {
        const bool pin = fits(used, c);
        HIP_CHECK(hipMemcpyAsync(pin ? p + used : c.dst, c.src, c.bytes, hipMemcpyDeviceToHost, l.stream));
        if (pin) used += step(c);
    }
    HIP_CHECK(hipStreamSynchronize(l.stream));
    used = 0;
    for (const HostCopy& c : copies) {
        if (!fits(used, c)) continue;
        std::memcpy(c.dst, p + used, c.bytes);
        used += step(c);
    }
}

size_t device_cache_release_all() {
    Cache& c = cache();
    std::lock_guard<std::mutex> lock(c.mu);
    int cur = 0;
    (void)hipGetDevice(&cur);
    size_t freed = 0;
    for (auto& kv : c.free_blocks) {
        if (kv.second.empty()) continue;
        if (hipSetDevice(kv.first) != hipSuccess) continue;
        (void)hipDeviceSynchronize();
        freed += drop_device(c, kv.first);
    }
    for (auto& kv : c.lanes) {
        if (kv.second.empty() || hipSetDevice(kv.first) != hipSuccess) continue;
        for (const Lane& l : kv.second) destroy_lane(l);
        kv.second.clear();
    }
    (void)hipSetDevice(cur);
    return freed;
}

size_t device_cache_bytes() {
    Cache& c = cache();
    std::lock_guard<std::mutex> lock(c.mu);
    size_t b = 0;
    for (auto& kv : c.cached) b += kv.second;
    return b;
}

}  // namespace egt
