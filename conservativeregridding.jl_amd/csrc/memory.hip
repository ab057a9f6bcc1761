// memory.hip -- the library's device memory: blocks that outlive the object that
// allocated them.
//
// A build allocates about 75 buffers.  Taken from the driver's stream-ordered
// pool and given back each time they cost more than the build's kernels: the
// pool unmaps large blocks when they are freed (5.5 + 2.2 ms for one quarter
// degree regridder, whatever its release threshold) and maps them again at the
// next build.  So freed blocks are kept here and handed out again:
//
//   * a block freed in order on a stream (a temporary) serves the next
//     allocation on that stream at once, as a stream-ordered pool would;
//   * a block owned by a handle (any stream may still be using it when the
//     handle is destroyed) serves again only after a device synchronisation,
//     made when such a block is first wanted: one per build in a loop of builds;
//   * a temporary of another stream is left to that stream: the allocation gets
//     a new block, so threads that build on their own streams do not wait for
//     one another;
//   * the kept blocks are bounded (1/64 of the device's memory: 4.5 GB); past
//     that, and for blocks no allocation has taken over the last kKeep frees,
//     the oldest go back to the driver, and all of them when an allocation fails.
//
// A build from host inputs and one field there and back: quarter degree ->
// HEALPix 256 21.6 -> 7.9 ms, 1 degree -> C48 3.0 -> 1.8 ms, 4 -> 5 degrees
// 2.2 -> 1.1 ms; the reverse mode's temporaries 0.42 -> 0.37 ms (C96 -> 1 degree).
#include <unistd.h>

#include <cstring>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "common.hpp"

namespace cr {

namespace {

constexpr uint64_t kKeep = 4096;  // frees a block may wait for its next use

enum State { kClean, kOnStream, kUnknown };  // who may still be using a free block: nobody, `stream`, anybody

struct Free {
    void *p;
    State state;
    hipStream_t stream;
    bool pool;       // from hipMallocAsync
    uint64_t stamp;  // number of frees when it was freed
};

struct Live {
    size_t bytes;
    int device;
    bool pool;
};

struct Device {
    std::multimap<size_t, Free> free;  // by size
    size_t kept = 0, cap = 0;
    uint64_t frees = 0;
};

struct Cache {
    std::mutex mu;
    std::unordered_map<void *, Live> live;
    std::map<int, Device> devices;
    pid_t pid = getpid();
};

// never destroyed: handles may be released while the process ends
Cache &cache() {
    static Cache *c = new Cache;
    return *c;
}

// sizes in steps of an eighth, so that nearly equal requests share blocks
size_t rounded(size_t bytes) {
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

bool synchronise(Device &d) {
    if (hipDeviceSynchronize() != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    for (auto &f : d.free) f.second.state = kClean;
    return true;
}

// Give blocks back to the driver until `most` bytes are kept; those older than
// `before` in any case.  The caller has made the device current.
void trim(Device &d, size_t most, uint64_t before) {
    bool synced = false;
    while (!d.free.empty()) {
        auto oldest = d.free.begin();
        for (auto it = d.free.begin(); it != d.free.end(); ++it)
            if (it->second.stamp < oldest->second.stamp) oldest = it;
        if (d.kept <= most && oldest->second.stamp >= before) return;
        if (!synced && !(synced = synchronise(d))) return;
        d.kept -= oldest->first;
        if (oldest->second.pool) (void)hipFreeAsync(oldest->second.p, nullptr);
        else (void)hipFree(oldest->second.p);
        d.free.erase(oldest);
    }
}

// The smallest free block of `bytes` that `ok` accepts and that is not much larger.
template <class F>
std::multimap<size_t, Free>::iterator find(Device &d, size_t bytes, F ok) {
    const size_t most = bytes + bytes / 4 + 4096;
    for (auto it = d.free.lower_bound(bytes); it != d.free.end() && it->first <= most; ++it)
        if (ok(it->second)) return it;
    return d.free.end();
}

}  // namespace

// `ordered`: the memory is first used on stream s; else on any stream.
void *device_alloc(size_t bytes, bool ordered, hipStream_t s) {
    int dev = 0;
    CR_HIP(hipGetDevice(&dev));
    const size_t want = rounded(bytes);
    Cache &c = cache();
    std::lock_guard<std::mutex> lock(c.mu);
    Device &d = c.devices[dev];
    if (!d.cap) {
        size_t avail = 0, total = 0;
        CR_HIP(hipMemGetInfo(&avail, &total));
        d.cap = total / 64;
        hipMemPool_t pool;
        uint64_t thr = UINT64_MAX;
        if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess)
            (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &thr);
    }
    auto usable = [&](const Free &f) {
        return f.state == kClean || (f.state == kOnStream && ordered && f.stream == s);
    };
    auto it = find(d, want, usable);
    if (it == d.free.end() && find(d, want, [](const Free &f) { return f.state == kUnknown; }) != d.free.end() &&
        synchronise(d))
        it = find(d, want, usable);
    if (it != d.free.end()) {
        void *p = it->second.p;
        c.live[p] = {it->first, dev, it->second.pool};
        d.kept -= it->first;
        d.free.erase(it);
        return p;
    }
    auto fresh = [&](void **p) { return ordered ? hipMallocAsync(p, want, s) : hipMalloc(p, want); };
    void *p = nullptr;
    hipError_t e = fresh(&p);
    if (e == hipErrorOutOfMemory && !d.free.empty()) {
        (void)hipGetLastError();
        trim(d, 0, UINT64_MAX);
        (void)hipDeviceSynchronize();
        e = fresh(&p);
    }
    CR_HIP(e);
    c.live[p] = {want, dev, ordered};
    return p;
}

// `ordered`: every use of the memory is in order on stream s; else unknown.
void device_free(void *p, bool ordered, hipStream_t s) {
    if (!p) return;
    Cache &c = cache();
    if (getpid() != c.pid) return;  // a forked child owns no device memory (and the lock may be held forever)
    std::lock_guard<std::mutex> lock(c.mu);
    auto l = c.live.find(p);
    if (l == c.live.end()) return;
    const Live b = l->second;
    c.live.erase(l);
    Device &d = c.devices[b.device];
    d.free.insert({b.bytes, Free{p, ordered ? kOnStream : kUnknown, s, b.pool, d.frees++}});
    d.kept += b.bytes;
    const uint64_t before = d.frees > kKeep ? d.frees - kKeep : 0;
    if (d.kept > d.cap || (before && d.frees % 64 == 0)) {
        int dev = b.device;
        if (hipGetDevice(&dev) != hipSuccess) return;
        if (dev != b.device && hipSetDevice(b.device) != hipSuccess) return;
        trim(d, d.cap, before);
        if (dev != b.device) (void)hipSetDevice(dev);
    }
}

}  // namespace cr
