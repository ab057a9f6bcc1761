// memory.hip on the host, over a runtime that only notes what it is asked to do.
#include <condition_variable>
#include <cstdlib>
#include <memory>
#include <set>

#include "../conservativeregridding.jl_amd/csrc/memory.hip"

namespace {
std::mutex g_mu;
std::condition_variable g_cv;
std::string g_log;
std::set<void *> g_capturing;
size_t g_total = (size_t)64 << 20, g_used = 0, g_room = ~(size_t)0;
bool g_hold = false, g_holding = false;  // driver allocations stop until released
std::unordered_map<void *, size_t> g_size;
void note(const std::string &s) {
    std::lock_guard<std::mutex> l(g_mu);
    g_log += s + ";";
}
thread_local hipStreamCaptureMode t_mode = hipStreamCaptureModeGlobal;
hipError_t get(void **p, size_t n) {
    std::unique_lock<std::mutex> l(g_mu);
    if (g_hold) {
        g_holding = true;
        g_cv.notify_all();
        g_cv.wait(l, [] { return !g_hold; });
        g_holding = false;
    }
    if (g_used + n > g_room) return hipErrorOutOfMemory;
    *p = std::malloc(16);
    g_size[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t put(void *p) {
    std::lock_guard<std::mutex> l(g_mu);
    g_used -= g_size.at(p);
    g_size.erase(p);
    return hipSuccess;  // (not freed: addresses stay unique)
}
std::string name(const void *s) { return std::to_string((size_t)s); }
thread_local std::unique_ptr<cr::CallScope> t_scope;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemGetInfo(size_t *a, size_t *t) { return *a = *t = g_total, hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *, int) { return hipErrorUnknown; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { return std::swap(*m, t_mode), hipSuccess; }
void strict(const char *call) {  // these break captures of other modes
    if (t_mode != hipStreamCaptureModeRelaxed) note(std::string(call) + " in another mode than relaxed");
}
hipError_t hipMalloc(void **p, size_t n) { return strict("malloc"), note("malloc"), get(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) { return note("malloc@" + name(s)), get(p, n); }
hipError_t hipFree(void *p) { return strict("free"), note("free"), put(p); }
hipError_t hipFreeAsync(void *p, hipStream_t s) { return note("free@" + name(s)), put(p); }
hipError_t hipDeviceSynchronize(void) { return note("devicesync"), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return note("sync@" + name(s)), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    std::lock_guard<std::mutex> l(g_mu);
    return *st = g_capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}

void call_begin(void) { t_scope.reset(new cr::CallScope); }
void call_fail(void) { t_scope->failed = true; }
void call_end(void) { t_scope.reset(); }
// use: 0 temporary, 1 kept, 2 any stream; null: refused or out of memory
void *mem_alloc(size_t n, int use, void *s) {
    try {
        return cr::device_alloc(n, (cr::Memory)use, (hipStream_t)s);
    } catch (const cr::Error &e) {
        note("error" + std::to_string((int)e.status));
        return nullptr;
    }
}
void mem_free(void *p, void *s) { cr::device_free(p, true, (hipStream_t)s); }
void mem_sync(void *s) { cr::synchronise((hipStream_t)s); }
// a handle's buffer, the handle used on streams (Uses bits)
void handle_free(void *p, unsigned bits) {
    cr::Uses u;
    u.bits = bits;
    cr::ReleaseScope as(u);
    cr::device_free(p, false, nullptr);
}
void set_capturing(void *s, int on) {
    if (on) g_capturing.insert(s);
    else g_capturing.erase(s);
}
void set_room(size_t n) { g_room = n; }
size_t used(void) { return g_used; }
void hold(int on) {
    std::lock_guard<std::mutex> l(g_mu);
    g_hold = on;
    g_cv.notify_all();
}
int wait_held(void) {
    std::unique_lock<std::mutex> l(g_mu);
    return g_cv.wait_for(l, std::chrono::seconds(20), [] { return g_holding; });
}
size_t take_log(char *to, size_t n) {
    std::lock_guard<std::mutex> l(g_mu);
    const size_t m = std::min(n - 1, g_log.size());
    g_log.copy(to, m);
    to[m] = 0;
    g_log.clear();
    return m;
}
}
namespace cr {
void set_error(const std::string &) {}
}
