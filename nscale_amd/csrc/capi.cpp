// Library-level C entry points: errors, init, and the thin operator wrappers whose
// implementations live in the kernel translation units.
#include <algorithm>
#include <atomic>
#include <cstdarg>
#include <cstring>
#include <mutex>

#include "common.hpp"

namespace nsc {

static thread_local char g_err[512] = {0};

void set_error(const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}
void clear_error() { g_err[0] = 0; }

namespace {
struct SyncState {
    bool blocking = false;
    hipEvent_t ev = nullptr;
    ~SyncState() {
        if (ev) (void)hipEventDestroy(ev);
    }
};
SyncState& sync_state() {
    static thread_local SyncState st;
    return st;
}
}  // namespace

void set_thread_blocking_sync(bool on) { sync_state().blocking = on; }

namespace {
// per-thread pinned word and event for the pass loops' asynchronous count reads
struct CountReader {
    int* host = nullptr;
    hipEvent_t ev = nullptr;
    int dev = -1;
    bool bridge = true;
    bool failed = false;
    ~CountReader() {
        if (ev) (void)hipEventDestroy(ev);
        if (host) (void)hipHostFree(host);
    }
};
CountReader& count_reader() {
    static thread_local CountReader r;
    return r;
}
}  // namespace

bool& thread_serving() {
    static thread_local bool serving = false;
    return serving;
}

bool set_thread_pass_bridge(bool on) {
    const bool prev = count_reader().bridge;
    count_reader().bridge = on;
    return prev;
}

int* count_read_async(const int* d, hipStream_t s) {
    CountReader& r = count_reader();
    if (!r.bridge || r.failed) return nullptr;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    if (!r.host && hipHostMalloc(reinterpret_cast<void**>(&r.host), 64, hipHostMallocDefault) != hipSuccess) {
        r.host = nullptr;
        r.failed = true;
        (void)hipGetLastError();
        return nullptr;
    }
    if (!r.ev || r.dev != dev) {
        if (r.ev) (void)hipEventDestroy(r.ev);
        r.ev = nullptr;
        if (hipEventCreateWithFlags(&r.ev, hipEventDisableTiming) != hipSuccess) {
            r.ev = nullptr;
            r.failed = true;
            (void)hipGetLastError();
            return nullptr;
        }
        r.dev = dev;
    }
    if (hipMemcpyAsync(r.host, d, sizeof(int), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipEventRecord(r.ev, s) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    return r.host;
}

hipError_t count_wait() { return hipEventSynchronize(count_reader().ev); }

Arena*& thread_arena() {
    static thread_local Arena* a = nullptr;
    return a;
}

// ---- the call cache --------------------------------------------------------------------------
// Up to kCacheSlots blocks per thread.  A call (from its first live scratch buffer to the release of
// its last) holds one block, used as a stack, and leaves an event behind its work on its stream.  The
// next call takes a block whose event has passed, or one last used on its own stream after making the
// stream wait for that event (work queued there is ahead of it anyway; the wait also covers a handle
// that names another stream by now).  A block still in use on another stream is left alone, so calls on
// different streams overlap as before; with no block free, and for streams under capture (the captured
// work would run again later, when the block may be someone else's), the pool serves.
// Bounds: kCacheBlock bytes a block, kCacheTotal over all threads.  Blocks come from the pool and
// return to it when they are outgrown, when none of kCacheWindow calls needed a quarter of one, and when
// the thread ends.
namespace {
constexpr int kCacheSlots = 4, kCacheWindow = 64;
constexpr size_t kCacheBlock = (size_t)1 << 30, kCacheTotal = (size_t)4 << 30, kCacheStep = (size_t)2 << 20;
std::atomic<size_t> g_cache_bytes{0};

struct CacheSlot {
    Arena arena;
    hipEvent_t done = nullptr;  // behind the last call's work
    hipStream_t stream = nullptr;
    int dev = -1;
    bool pending = false;  // `done` has been recorded and not yet seen complete
    size_t want = 0;       // bytes the last call that did not fit would have needed
    size_t recent = 0;     // most bytes a call needed in the current window
    int calls = 0;         // calls in the current window
};

struct CallCache {
    CacheSlot slots[kCacheSlots];
    CacheSlot* cur = nullptr;  // the current call's block
    int live = 0;              // its buffers not yet released
    size_t peak = 0, missed = 0;
    ~CallCache() {
        for (CacheSlot& c : slots) {
            if (c.pending) (void)hipEventSynchronize(c.done);
            if (c.done) (void)hipEventDestroy(c.done);
            if (c.arena.base) {
                (void)hipFreeAsync(c.arena.base, nullptr);  // its last use is over
                g_cache_bytes -= c.arena.cap;
            }
        }
        (void)hipGetLastError();
    }
};
CallCache& call_cache() {
    static thread_local CallCache c;
    return c;
}

bool slot_idle(CacheSlot& c) {
    if (!c.pending) return true;
    if (hipEventQuery(c.done) != hipSuccess) {
        (void)hipGetLastError();  // not ready is an answer here, not an error
        return false;
    }
    c.pending = false;
    return true;
}

// the block of a call on stream s, ordered behind the block's last use; nullptr: none is free
CacheSlot* pick_slot(CallCache& C, int dev, hipStream_t s) {
    CacheSlot *idle = nullptr, *fresh = nullptr;
    for (CacheSlot& c : C.slots) {
        if (c.dev < 0) {
            if (!fresh) fresh = &c;
            continue;
        }
        if (c.dev != dev) continue;
        if (c.stream == s) {
            if (!slot_idle(c) && hipStreamWaitEvent(s, c.done, 0) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
            return &c;
        }
        if (!idle && slot_idle(c)) idle = &c;
    }
    if (idle) return idle;
    if (!fresh) return nullptr;
    if (hipEventCreateWithFlags(&fresh->done, hipEventDisableTiming) != hipSuccess) {
        fresh->done = nullptr;
        (void)hipGetLastError();
        return nullptr;
    }
    fresh->dev = dev;
    return fresh;
}

// resizes an ordered block to `cap` bytes (0: none)
void resize_block(CacheSlot& c, size_t cap, hipStream_t s) {
    if (c.arena.base) {
        (void)hipFreeAsync(c.arena.base, s);
        g_cache_bytes -= c.arena.cap;
        c.arena = Arena();
    }
    if (!cap) return;
    if (g_cache_bytes.fetch_add(cap) + cap > kCacheTotal) {
        g_cache_bytes -= cap;
        return;
    }
    void* p = nullptr;
    if (hipMallocAsync(&p, cap, s) != hipSuccess) {
        (void)hipGetLastError();
        g_cache_bytes -= cap;
        return;
    }
    c.arena.base = static_cast<uint8_t*>(p);
    c.arena.cap = cap;
}
size_t block_size(size_t bytes) { return (bytes + bytes / 8 + kCacheStep) / kCacheStep * kCacheStep; }
}  // namespace

void* call_cache_take(size_t bytes, hipStream_t s) {
    CallCache& C = call_cache();
    if (C.live == 0) {
        hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
        if (bytes > kCacheBlock) return nullptr;
        if (hipStreamIsCapturing(s, &st) != hipSuccess || st != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            return nullptr;
        }
        // a block belongs to the stream's device, its event to the current one: serve where they agree
        int dev = 0, sdev = 0;
        if (hipGetDevice(&dev) != hipSuccess || (s && hipStreamGetDevice(s, &sdev) != hipSuccess) || (s && sdev != dev)) {
            (void)hipGetLastError();
            return nullptr;
        }
        CacheSlot* c = pick_slot(C, dev, s);
        if (!c) return nullptr;
        c->stream = s;
        if (++c->calls >= kCacheWindow) {
            if (c->arena.cap > 4 * c->recent && c->arena.cap > 32 * kCacheStep) resize_block(*c, block_size(2 * c->recent), s);
            c->calls = 0;
            c->recent = 0;
        }
        const size_t want = std::min(std::max(bytes, c->want), kCacheBlock);
        c->want = 0;
        if (want > c->arena.cap) resize_block(*c, std::min(block_size(want), kCacheBlock), s);
        C.cur = c;
        C.peak = C.missed = 0;
    } else if (C.cur->stream != s) {
        return nullptr;
    }
    void* p = C.cur->arena.take(bytes);
    if (p) {
        ++C.live;
        C.peak = std::max(C.peak, C.cur->arena.top);
    } else {
        C.missed += bytes + 512;
        if (C.live == 0) C.cur = nullptr;
    }
    return p;
}

void call_cache_give(void* p) {
    CallCache& C = call_cache();
    CacheSlot& c = *C.cur;
    (void)c.arena.give(p);
    if (--C.live > 0) return;
    const size_t need = C.peak + C.missed;
    if (C.missed) c.want = need;
    c.recent = std::max(c.recent, need);
    c.pending = true;
    if (hipEventRecord(c.done, c.stream) != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamSynchronize(c.stream);
        c.pending = false;
    }
    C.cur = nullptr;
}

hipError_t stream_sync(hipStream_t s) {
    SyncState& st = sync_state();
    if (!st.blocking) return hipStreamSynchronize(s);
    if (!st.ev) {
        const hipError_t e = hipEventCreateWithFlags(&st.ev, hipEventBlockingSync | hipEventDisableTiming);
        if (e != hipSuccess) return e;
    }
    hipError_t e = hipEventRecord(st.ev, s);
    if (e != hipSuccess) return e;
    e = hipEventSynchronize(st.ev);
    if (e != hipSuccess) return e;
    // the work is done; this returns at once and completes any pageable host copy bookkeeping
    return hipStreamSynchronize(s);
}

int ensure_init() {
    static std::once_flag once;
    static int status = NSC_OK;
    std::call_once(once, [] {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) {
            set_error("no HIP device: %s", hipGetErrorString(e));
            status = NSC_ERR_HIP;
            return;
        }
        hipMemPool_t pool;
        if (hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess) {
            uint64_t thr = UINT64_MAX;
            (void)hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &thr);
        }
    });
    return status;
}

}  // namespace nsc

using namespace nsc;

extern "C" {

const char* nsc_version(void) { return "nscale_amd 0.1 (gfx950)"; }
const char* nsc_last_error(void) { return g_err; }
int nsc_init(void) { return ensure_init(); }

int nsc_imreconstruct_u8(const uint8_t* marker, const uint8_t* mask, uint8_t* out, int w, int h, int conn,
                         void* stream) {
    NSC_ARG(marker && mask && out && w > 0 && h > 0 && valid_conn(conn), "imreconstruct_u8");
    NSC_CHECK(ensure_init());
    return recon_impl<uint8_t>(marker, mask, out, w, h, conn, as_stream(stream));
}

int nsc_imreconstruct_f32(const float* marker, const float* mask, float* out, int w, int h, int conn,
                          void* stream) {
    NSC_ARG(marker && mask && out && w > 0 && h > 0 && valid_conn(conn), "imreconstruct_f32");
    NSC_CHECK(ensure_init());
    return recon_impl<float>(marker, mask, out, w, h, conn, as_stream(stream));
}

int nsc_imreconstruct_u8_batched(const nsc_recon_desc* descs, int n, void* stream) {
    NSC_ARG(descs && n > 0, "imreconstruct_u8_batched");
    NSC_CHECK(ensure_init());
    return recon_batched_impl<uint8_t>(descs, n, as_stream(stream));
}

int nsc_imreconstruct_f32_batched(const nsc_recon_desc* descs, int n, void* stream) {
    NSC_ARG(descs && n > 0, "imreconstruct_f32_batched");
    NSC_CHECK(ensure_init());
    return recon_batched_impl<float>(descs, n, as_stream(stream));
}

int nsc_imreconstruct_i32(const int32_t* marker, const int32_t* mask, int32_t* out, int w, int h, int conn,
                          void* stream) {
    NSC_ARG(marker && mask && out && w > 0 && h > 0 && valid_conn(conn), "imreconstruct_i32");
    NSC_CHECK(ensure_init());
    return recon_impl<int32_t>(marker, mask, out, w, h, conn, as_stream(stream));
}

}  // extern "C"
