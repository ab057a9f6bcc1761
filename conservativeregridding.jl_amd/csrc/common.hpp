// common.hpp -- shared definitions of the HIP library (host + device).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/crhip.h"

#define CR_HD __host__ __device__ __forceinline__

namespace cr {

// ------------------------------------------------------------- errors --
void set_error(const std::string &msg);

struct Error {
    cr_status status;
    std::string msg;
};

#define CR_HIP(expr)                                                                     \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess)                                                            \
            throw ::cr::Error{e_ == hipErrorOutOfMemory ? CR_OUT_OF_MEMORY : CR_HIP_ERROR, \
                              std::string(#expr) + ": " + hipGetErrorString(e_)};        \
    } while (0)

#define CR_REQUIRE(cond, status, msg)                               \
    do {                                                            \
        if (!(cond)) throw ::cr::Error{(status), std::string(msg)}; \
    } while (0)

// True while `s` is being captured into a HIP graph.  Lazy per-regridder set-up
// (tile plans, long-row lists, the default variant) allocates, copies to the
// host and synchronises: none of that may run inside a capture.
inline bool stream_capturing(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();  // e.g. the legacy null stream during a global capture
        return true;
    }
    return st != hipStreamCaptureStatusNone;
}

#define CR_REQUIRE_NOT_CAPTURING(s, what)                                                                \
    CR_REQUIRE(!::cr::stream_capturing(s), CR_UNSUPPORTED,                                               \
               std::string(what) + " is not made yet and cannot be made during stream capture: call "   \
                                   "cr_regrid_prepare (or one cr_regrid) with the same arguments first")

// Calls that allocate and synchronise whatever was prepared: refused before they
// enqueue anything, so that the capture goes on without them.  (The null stream is
// never captured; other captures do not concern it.)
inline void refuse_capture(hipStream_t s, const char *call) {
    CR_REQUIRE(!s || !stream_capturing(s), CR_UNSUPPORTED,
               std::string(call) + " allocates device memory and synchronises its stream: it cannot run while that "
                                   "stream is being captured");
}

// Device memory (memory.hip keeps freed blocks for the next allocation and says
// who gets which).
enum Memory {
    kTemporary,  // used and freed in order on its stream, within one library call
    kKept,       // owned by a handle: first used in order on its stream, then on any
    kAnyStream   // owned by a handle: used on any stream from the start
};
void *device_alloc(size_t bytes, Memory use, hipStream_t s);
void device_free(void *p, bool ordered, hipStream_t s);  // ordered: a temporary's

// One library call on this thread (guard() holds one).
struct CallScope {
    CallScope();
    ~CallScope();
    CallScope(const CallScope &) = delete;
    bool failed = false;  // it may have left its handles' work pending
};
// Wait for stream s: what this call has freed in order on it so far is free for anyone.
void synchronise(hipStream_t s);

// The streams on which a handle may have work pending: marked by every call that
// returns without synchronising its stream.
struct Uses {
    static constexpr unsigned kOnNull = 1, kElsewhere = 2;
    mutable std::atomic<unsigned> bits{0};
    void on(hipStream_t s) const {
        const unsigned b = s ? kElsewhere : kOnNull;
        if (!(bits.load(std::memory_order_relaxed) & b)) bits.fetch_or(b);
    }
};
// Buffers of a handle released on this thread in its lifetime are free once the
// work those uses left pending is done.
struct ReleaseScope {
    explicit ReleaseScope(const Uses &u);
    ~ReleaseScope();
    ReleaseScope(const ReleaseScope &) = delete;
};

// DevBuf(n): kAnyStream; DevBuf(n, stream): kTemporary; alloc_kept(n, stream): kKept.
template <class T>
struct DevBuf {
    T *p = nullptr;
    size_t n = 0;
    hipStream_t st = nullptr;
    bool ordered = false;  // freed in order on st
    DevBuf() = default;
    explicit DevBuf(size_t count) { alloc(count); }
    DevBuf(size_t count, hipStream_t s) { alloc_async(count, s); }
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : p(o.p), n(o.n), st(o.st), ordered(o.ordered) {
        o.p = nullptr;
        o.n = 0;
    }
    DevBuf &operator=(DevBuf &&o) noexcept {
        if (this != &o) {
            release();
            p = o.p; n = o.n; st = o.st; ordered = o.ordered;
            o.p = nullptr; o.n = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    void alloc(size_t count) { get(count, kAnyStream, nullptr); }
    void alloc_async(size_t count, hipStream_t s) { get(count, kTemporary, s); }
    void alloc_kept(size_t count, hipStream_t s) { get(count, kKept, s); }
    void release() {
        device_free(p, ordered, st);
        p = nullptr;
        n = 0;
    }
    size_t bytes() const { return n * sizeof(T); }

  private:
    void get(size_t count, Memory use, hipStream_t s) {
        release();
        st = s;
        ordered = use == kTemporary;
        if (count) p = (T *)device_alloc(count * sizeof(T), use, s);
        n = count;
    }
};

// Free temporaries (in order on their stream).
template <class... T>
void release(DevBuf<T> &...b) {
    (b.release(), ...);
}

// Run a body and turn exceptions into a status + thread-local message.
template <class F>
cr_status guard(F &&f) {
    CallScope call;
    try {
        f();
        return CR_OK;
    } catch (const Error &e) {
        call.failed = true;
        set_error(e.msg);
        return e.status;
    } catch (const std::bad_alloc &) {
        call.failed = true;
        set_error("host allocation failed");
        return CR_OUT_OF_MEMORY;
    } catch (const std::exception &e) {
        call.failed = true;
        set_error(e.what());
        return CR_INTERNAL;
    }
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

inline void check_device() {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n == 0) throw Error{CR_NO_DEVICE, "no HIP device is visible"};
}

// Widest cell polygon a grid may hold (vertices per cell).
constexpr int kMaxCellVertices = 64;

inline unsigned grid_for(int64_t n, int block) {
    int64_t g = (n + block - 1) / block;
    return (unsigned)(g < 1 ? 1 : g);
}

}  // namespace cr

// ------------------------------------------------------------- handles --
struct cr_grid {
    cr::Uses uses;
    int64_t ncells = 0;
    int32_t nv = 0;
    int32_t convex = 0;
    int32_t flipped = 0;
    int64_t nverts = 0;          // caller-visible vertices (points of a point grid)
    cr::DevBuf<double> cells;    // ncells * nv * 3, xyz interleaved per vertex
    cr::DevBuf<int32_t> vidx;    // ncells * nv: caller vertex of each cell slot
    int32_t private_vertices = 0;  // 1: no vertex index is shared by two cells (tables of cells)
    cr::DevBuf<int32_t> fold;    // 2 * nfold: (primary, partner) cells of a folded row
    int64_t nfold = 0;
    // Planar manifold: the caller's vertices (nverts * 2, x and y); `cells`
    // then holds their gnomonic images on the unit sphere, which only the
    // candidate search reads (straight edges map to great-circle arcs)
    int32_t planar = 0;
    cr::DevBuf<double> xy;
};
