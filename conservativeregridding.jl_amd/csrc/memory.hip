// memory.hip -- the library's device memory: blocks that outlive the object that
// allocated them.
//
// A build allocates about 75 buffers.  Taken from the driver's stream-ordered
// pool and given back each time they cost more than the build's kernels: the
// pool unmaps large blocks when they are freed (5.5 + 2.2 ms for one quarter
// degree regridder, whatever its release threshold) and maps them again at the
// next build.  So freed blocks are kept here and handed out again, by who may
// still be using them:
//
//   * kCall: a temporary of a library call that still runs serves that call's next
//     allocation on its stream at once, as a stream-ordered pool would, and nobody
//     else.  Once the call has synchronised that stream it is clean (what it frees
//     after its last synchronise() costs another one at its end).  A stream's handle
//     says nothing between calls: hipStreamPerThread is another stream on every
//     thread, and a handle may come back for a new stream.  Only the null stream is
//     always the same one: its temporaries become kNull without a synchronisation;
//   * kNull: pending work on the null stream only (also a handle's blocks that was
//     used on no other stream): serves the next allocation in order on that stream,
//     and any new handle's buffer once the null stream is synchronised;
//   * kUnknown: a handle that was used on another stream, possibly by a graph: its
//     blocks serve a new handle's buffers once the device's pending work is done.
//     The allocation waits for that by hipFree of a small block, which synchronises
//     the device by contract; hipDeviceSynchronize would break every stream capture
//     in progress, on whatever thread and in whatever mode.  Temporaries do not
//     wait, so calls that only need those stay ordered by their own stream;
//   * kClean: nobody.
//
// The driver's allocations and frees are asked for in the relaxed capture mode: a
// handle may be released (by a garbage collector) while some stream, its thread's own
// too, is being captured.  No lock is held while the driver works.  The kept blocks are bounded (1/64 of the
// device's memory: 4.5 GB): past that the oldest go back to the driver until a quarter
// of the bound is free, and so do blocks that no allocation took over the last kKeep
// frees, and all of them when an allocation fails.
//
// A build from host inputs and one field there and back: quarter degree ->
// HEALPix 256 21.6 -> 7.9 ms, 1 degree -> C48 3.0 -> 1.8 ms, 4 -> 5 degrees
// 2.2 -> 1.1 ms; the reverse mode's temporaries 0.42 -> 0.37 ms (C96 -> 1 degree).
#include <pthread.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "common.hpp"

namespace cr {

namespace {

constexpr uint64_t kKeep = 4096;  // frees a block may wait for its next use

enum State { kClean, kNull, kCall, kUnknown };

struct Free {
    void *p;
    State state;
    uint64_t call;  // kCall: the call and the stream it was freed in order on
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
    uint64_t calls = 0;
};

// A forked child owns no device memory, and the lock may be held forever there.
std::atomic<bool> g_child{false};

// never destroyed: handles may be released while the process ends
Cache &cache() {
    static Cache *c = [] {
        pthread_atfork(nullptr, nullptr, [] { g_child = true; });
        return new Cache;
    }();
    return *c;
}

// The library call of this thread, and how a handle's buffers are released.
struct Call {
    int depth = 0;
    uint64_t id = 0;     // 0: no temporaries yet
    size_t pending = 0;  // its free blocks in state kCall
    bool checked = false;
    hipStream_t checked_stream = nullptr;  // not capturing
};
thread_local Call t_call;
thread_local State t_release = kUnknown;

using Lock = std::unique_lock<std::mutex>;

// sizes in steps of an eighth, so that nearly equal requests share blocks
size_t rounded(size_t bytes) {
    size_t step = 512;
    while (step * 16 <= bytes) step *= 2;
    return (bytes + step - 1) / step * step;
}

// In its lifetime this thread's hipMalloc and hipFree disturb no capture.
struct Relaxed {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
    ~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// Wait for the device's pending work (the caller has made it current).  No lock held.
bool device_wait() {
    Relaxed r;
    void *p = nullptr;
    if (hipMalloc(&p, 256) == hipSuccess && hipFree(p) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

// The smallest free block of `bytes` that `ok` accepts and that is not much larger.
template <class F>
std::multimap<size_t, Free>::iterator find(Device &d, size_t bytes, F ok) {
    const size_t most = bytes + bytes / 4 + 4096;
    for (auto it = d.free.lower_bound(bytes); it != d.free.end() && it->first <= most; ++it)
        if (ok(it->second)) return it;
    return d.free.end();
}

// Wait without the lock until the free blocks in state st are clean.
bool wait_and_clean(Device &d, State st, Lock &lock) {
    const uint64_t now = d.frees;
    lock.unlock();
    const bool done = st == kNull ? hipStreamSynchronize(nullptr) == hipSuccess : device_wait();
    if (!done) (void)hipGetLastError();
    lock.lock();
    if (done)
        for (auto &f : d.free)
            if (f.second.stamp < now && f.second.state == st) f.second.state = kClean;
    return done;
}

// Give blocks back to the driver: the oldest until `most` bytes are kept, and those
// older than `before`.  Blocks of running calls stay, but for this thread's own when
// `own`.  The caller has made the device current and holds the lock.
void trim(Device &d, size_t most, uint64_t before, bool own, Lock &lock) {
    auto mine = [&](const Free &f) { return own && f.call && f.call == t_call.id; };
    std::vector<std::multimap<size_t, Free>::iterator> order;
    for (auto it = d.free.begin(); it != d.free.end(); ++it)
        if (it->second.state != kCall || mine(it->second)) order.push_back(it);
    std::sort(order.begin(), order.end(), [](auto a, auto b) { return a->second.stamp < b->second.stamp; });
    std::vector<std::pair<size_t, Free>> out;
    for (auto it : order) {
        if (d.kept <= most && it->second.stamp >= before) break;
        d.kept -= it->first;
        if (it->second.state == kCall) --t_call.pending;
        out.push_back(*it);
        d.free.erase(it);
    }
    if (out.empty()) return;
    lock.unlock();
    auto give = [](const Free &f) {
        if (f.pool) (void)hipFreeAsync(f.p, f.state == kCall ? f.stream : nullptr);
        else (void)hipFree(f.p);
    };
    Relaxed r;
    std::vector<std::pair<size_t, Free>> back;
    for (auto &b : out) {
        if (b.second.state == kUnknown) back.push_back(b);
        else give(b.second);
    }
    if (!back.empty() && device_wait()) {
        for (auto &b : back) give(b.second);
        back.clear();
    }
    (void)hipGetLastError();
    lock.lock();
    for (auto &b : back) {
        d.free.insert(b);
        d.kept += b.first;
    }
}

// Keep the bounds of device `index`, on whatever device this thread is.
void bound(Device &d, int index, Lock &lock) {
    const uint64_t before = d.frees > kKeep ? d.frees - kKeep : 0;
    const bool over = d.kept > d.cap;
    if (!over && !(before && d.frees % 64 == 0)) return;
    int dev = index;
    if (hipGetDevice(&dev) != hipSuccess) return;
    if (dev != index && hipSetDevice(index) != hipSuccess) return;
    trim(d, over ? d.cap / 4 * 3 : d.cap, before, false, lock);
    if (dev != index) (void)hipSetDevice(dev);
}

// Each block this call freed in order on its streams; f may give it another state.
template <class F>
void freed_by_call(Cache &c, F f) {
    if (!t_call.pending) return;
    for (auto &dev : c.devices)
        for (auto &b : dev.second.free)
            if (b.second.state == kCall && b.second.call == t_call.id) {
                f(b.second);
                if (b.second.state != kCall) --t_call.pending;
            }
}

// The call is over: synchronise the streams it freed temporaries on -- after a failure
// the null stream, too, for the sake of the handles it was reading.
void end_call(bool failed) {
    Cache &c = cache();
    std::vector<hipStream_t> pending;
    Lock lock(c.mu);
    freed_by_call(c, [&](Free &f) {
        if (!f.stream && !failed) f.state = kNull;
        else if (std::find(pending.begin(), pending.end(), f.stream) == pending.end()) pending.push_back(f.stream);
    });
    for (hipStream_t s : pending) {
        lock.unlock();
        const State st = hipStreamSynchronize(s) == hipSuccess ? kClean : kUnknown;
        if (st != kClean) (void)hipGetLastError();
        lock.lock();
        freed_by_call(c, [&](Free &f) {
            if (f.stream == s) f.state = st;
        });
    }
    for (auto &dev : c.devices) bound(dev.second, dev.first, lock);
}

}  // namespace

CallScope::CallScope() { ++t_call.depth; }

CallScope::~CallScope() {
    if (--t_call.depth) return;
    try {
        if (t_call.id && !g_child) end_call(failed);
    } catch (const std::exception &) {  // no host memory: the call's blocks stay its own
    }
    t_call = Call{};
}

void synchronise(hipStream_t s) {
    CR_HIP(hipStreamSynchronize(s));
    if (!t_call.pending) return;
    Cache &c = cache();
    Lock lock(c.mu);
    freed_by_call(c, [&](Free &f) {
        if (f.stream == s) f.state = kClean;
    });
}

ReleaseScope::ReleaseScope(const Uses &u) {
    const unsigned b = u.bits.load();
    t_release = b == 0 ? kClean : b == Uses::kOnNull ? kNull : kUnknown;
}
ReleaseScope::~ReleaseScope() { t_release = kUnknown; }

void *device_alloc(size_t bytes, Memory use, hipStream_t s) {
    const bool ordered = use != kAnyStream;
    int dev = 0;
    CR_HIP(hipGetDevice(&dev));
    // memory allocated while its stream is being captured would belong to the graph
    if (ordered && s && !(t_call.checked && t_call.checked_stream == s)) {
        refuse_capture(s, "this call");
        t_call.checked = t_call.depth > 0;
        t_call.checked_stream = s;
    }
    const size_t want = rounded(bytes);
    Cache &c = cache();
    CR_REQUIRE(!g_child, CR_HIP_ERROR, "a forked child has no device memory");
    Lock lock(c.mu);
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
    if (use == kTemporary && t_call.depth && !t_call.id) t_call.id = ++c.calls;
    auto usable = [&](const Free &f) {
        return f.state == kClean || (f.state == kNull && ordered && !s) ||
               (f.state == kCall && ordered && f.call == t_call.id && f.stream == s);
    };
    auto it = find(d, want, usable);
    for (State st : {kNull, kUnknown}) {
        if (it != d.free.end() || use == kTemporary) break;
        auto in_state = [st](const Free &f) { return f.state == st; };
        if (find(d, want, in_state) != d.free.end() && wait_and_clean(d, st, lock)) it = find(d, want, usable);
    }
    if (it != d.free.end()) {
        void *p = it->second.p;
        if (it->second.state == kCall) --t_call.pending;
        c.live[p] = {it->first, dev, it->second.pool};
        d.kept -= it->first;
        d.free.erase(it);
        return p;
    }
    lock.unlock();
    auto fresh = [&](void **p) {
        Relaxed r;
        return ordered ? hipMallocAsync(p, want, s) : hipMalloc(p, want);
    };
    void *p = nullptr;
    hipError_t e = fresh(&p);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        lock.lock();
        trim(d, 0, UINT64_MAX, true, lock);
        lock.unlock();
        (void)device_wait();
        e = fresh(&p);
    }
    CR_HIP(e);
    lock.lock();
    c.live[p] = {want, dev, ordered};
    return p;
}

void device_free(void *p, bool ordered, hipStream_t s) {
    if (!p) return;
    Cache &c = cache();
    if (g_child) return;
    try {
        Lock lock(c.mu);
        auto l = c.live.find(p);
        if (l == c.live.end()) return;
        const Live b = l->second;
        Device &d = c.devices[b.device];
        State st = t_release;
        if (ordered) st = t_call.id ? kCall : s ? kUnknown : kNull;
        d.free.insert({b.bytes, Free{p, st, st == kCall ? t_call.id : 0, s, b.pool, d.frees}});
        if (st == kCall) ++t_call.pending;
        c.live.erase(l);
        d.frees++;
        d.kept += b.bytes;
        bound(d, b.device, lock);
    } catch (const std::exception &) {  // no host memory for the list: the block is lost, not handed out twice
    }
}

}  // namespace cr
