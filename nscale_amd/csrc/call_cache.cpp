// The operators' scratch blocks that are kept between calls (see scratch.hpp).
//
// Up to kCacheSlots blocks per thread.  A call (from its first live scratch buffer to the release of
// its last) holds one block, used as a stack, and leaves an event behind its work on its stream.  The
// next call takes a block whose event has passed, or one last used on its own stream after making the
// stream wait for that event (work queued there is ahead of it anyway; the wait also covers a handle
// that names another stream by now).  A block still in use on another stream is left alone, so calls on
// different streams overlap as before; with no block free, and for streams under capture (the captured
// work would run again later, when the block may be someone else's), the pool serves.
// While any stream of the process is captured in global mode, asking an event whether it has passed, or
// waiting for it, counts as an unsafe call and would end that capture.  The events here are recorded on streams
// that are not captured and the answer only chooses a block, so the cache asks in relaxed mode.
// Bounds: kCacheBlock bytes a block, kCacheTotal over all threads.  Blocks come from the pool and
// return to it when they are outgrown, when none of kCacheWindow calls on one needed a quarter of it, when
// its thread's calls have passed it over kCacheAge times, when the thread ends, and, whichever thread
// holds them, when an allocation fails (a call that holds its block keeps it).  The lock of a thread's cache is for
// that last case; otherwise only its own thread takes it.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <vector>

#include "scratch.hpp"

namespace nsc {
namespace {
constexpr int kCacheSlots = 4, kCacheWindow = 64, kCacheAge = 2 * kCacheWindow;
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
    int passed = 0;        // calls of the thread since this block's last one
};

// relaxed capture mode of the calling thread while it lives
struct RelaxedCapture {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    bool set = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
    ~RelaxedCapture() {
        if (set) (void)hipThreadExchangeStreamCaptureMode(&mode);
    }
};

// returns a block whose last use is over to the pool, on no user's stream: on the null stream, or on a stream
// of its own while another one's capture forbids that
void free_block(void* p) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    hipStream_t own = nullptr;
    if (hipStreamIsCapturing(nullptr, &st) != hipSuccess &&
        hipStreamCreateWithFlags(&own, hipStreamNonBlocking) != hipSuccess)
        return;
    (void)hipFreeAsync(p, own);
    if (own) (void)hipStreamDestroy(own);
}

struct CallCache;
// every thread's cache (never destroyed: threads may end after the statics have)
struct Registry {
    std::mutex m;
    std::vector<CallCache*> caches;
};
Registry& registry() {
    static Registry* const r = new Registry;
    return *r;
}

struct CallCache {
    std::mutex m;
    CacheSlot slots[kCacheSlots];
    CacheSlot* cur = nullptr;  // the current call's block
    int live = 0;              // its buffers not yet released
    size_t peak = 0, missed = 0;
    CallCache() {
        Registry& r = registry();
        const std::lock_guard<std::mutex> lock(r.m);
        r.caches.push_back(this);
    }
    ~CallCache() {
        {
            Registry& r = registry();
            const std::lock_guard<std::mutex> lock(r.m);
            r.caches.erase(std::find(r.caches.begin(), r.caches.end(), this));
        }
        const RelaxedCapture relaxed;
        for (CacheSlot& c : slots) {
            if (c.pending) (void)hipEventSynchronize(c.done);
            if (c.done) (void)hipEventDestroy(c.done);
            if (c.arena.base) {
                free_block(c.arena.base);
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
    const RelaxedCapture relaxed;
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
// gives back, on stream s, the blocks of device dev that no call holds, over all threads; s waits for those
// whose work is still going on.  Whether there were any.
bool give_back_unused(int dev, hipStream_t s) {
    Registry& r = registry();
    const std::lock_guard<std::mutex> all(r.m);
    bool any = false;
    for (CallCache* C : r.caches) {
        const std::lock_guard<std::mutex> lock(C->m);
        for (CacheSlot& c : C->slots) {
            if (!c.arena.base || c.dev != dev || (C->live > 0 && &c == C->cur)) continue;
            if (!slot_idle(c) && hipStreamWaitEvent(s, c.done, 0) != hipSuccess) {
                (void)hipGetLastError();
                continue;
            }
            resize_block(c, 0, s);
            any = true;
        }
    }
    return any;
}

// one more call of the thread on another block: blocks that have been passed over for long go back
void age_blocks(CallCache& C, const CacheSlot* used, hipStream_t s) {
    for (CacheSlot& c : C.slots) {
        if (&c == used) c.passed = 0;
        else if (c.arena.base && ++c.passed >= kCacheAge && c.dev == used->dev && slot_idle(c)) resize_block(c, 0, s);
    }
}

// whether s is a stream of the current device, *dev, that is not being captured
bool plain_stream(hipStream_t s, int* dev) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    int sdev = 0;
    if (hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone && hipGetDevice(dev) == hipSuccess &&
        (!s || (hipStreamGetDevice(s, &sdev) == hipSuccess && sdev == *dev)))
        return true;
    (void)hipGetLastError();
    return false;
}
size_t block_size(size_t bytes) { return (bytes + bytes / 8 + kCacheStep) / kCacheStep * kCacheStep; }
}  // namespace

void* call_cache_take(size_t bytes, hipStream_t s) {
    CallCache& C = call_cache();
    const std::lock_guard<std::mutex> lock(C.m);
    if (C.live == 0) {
        // a block belongs to the stream's device, its event to the current one: serve where they agree
        int dev = 0;
        if (bytes > kCacheBlock || !plain_stream(s, &dev)) return nullptr;
        CacheSlot* c = pick_slot(C, dev, s);
        if (!c) return nullptr;
        c->stream = s;
        age_blocks(C, c, s);
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
    const std::lock_guard<std::mutex> lock(C.m);
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

hipError_t pool_alloc(void** p, size_t bytes, hipStream_t s) {
    hipError_t e = hipMallocAsync(p, bytes, s);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    int dev = 0;
    if (!plain_stream(s, &dev) || !give_back_unused(dev, s)) return e;
    e = hipMallocAsync(p, bytes, s);
    if (e == hipSuccess) return e;
    (void)hipGetLastError();
    // the freed blocks may be pieces that the pool holds on to: wait until they are free and let it return them
    const RelaxedCapture relaxed;
    hipMemPool_t pool;
    if (hipStreamSynchronize(s) == hipSuccess && hipDeviceGetDefaultMemPool(&pool, dev) == hipSuccess &&
        hipMemPoolTrimTo(pool, 0) == hipSuccess)
        e = hipMallocAsync(p, bytes, s);
    if (e != hipSuccess) (void)hipGetLastError();
    return e;
}

}  // namespace nsc
