// Stream-ordered scratch memory of the operators (host code only: the tests build it with a host compiler).
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "nscale_hip.h"

namespace nsc {

void set_error(const char* fmt, ...);

// Scratch comes from the calling thread's arena when one is active (a chain call activates its
// workspace's arena: a device buffer allocated once, handed out as a stack -- scopes nest, so
// frees arrive in reverse order, and a buffer freed out of order is reclaimed when everything
// above it is gone), else from the thread's call cache (below), else from the device's default memory
// pool (hipMallocAsync, release threshold raised at init).  Either way the memory is stream-ordered:
// reuse by a later operator on the same stream is safe without synchronisation.
struct Arena {
    uint8_t* base = nullptr;
    size_t cap = 0, top = 0;
    struct Entry { size_t off, end; bool live; };
    Entry stack[64];
    int depth = 0;
    void* take(size_t bytes) {
        const size_t off = (top + 255) & ~(size_t)255;
        if (!base || depth == 64 || off + bytes > cap) return nullptr;
        stack[depth++] = Entry{off, off + bytes, true};
        top = off + bytes;
        return base + off;
    }
    bool give(void* p) {
        if (!base || p < (void*)base || p >= (void*)(base + cap)) return false;
        const size_t off = (size_t)((uint8_t*)p - base);
        for (int k = depth - 1; k >= 0; --k)
            if (stack[k].off == off && stack[k].live) { stack[k].live = false; break; }
        while (depth > 0 && !stack[depth - 1].live) --depth;
        top = depth ? stack[depth - 1].end : 0;
        return true;
    }
};
Arena*& thread_arena();

// activates an arena for the calling thread for the lifetime of the guard
struct ArenaScope {
    Arena* prev;
    explicit ArenaScope(Arena* a) : prev(thread_arena()) { thread_arena() = a; }
    ~ArenaScope() { thread_arena() = prev; }
};

// Call cache: operator calls outside a chain take their scratch from blocks that the calling thread
// keeps (call_cache.cpp).  The pool's free and allocation cost 12-37 us a pair while one size repeats, and
// 360 us when sizes alternate (hipMallocAsync 200, hipFreeAsync 160; five pairs are one labelling
// call's), more than most operators' kernels.  take returns nullptr where the cache does not serve: the
// pool does then.
void* call_cache_take(size_t bytes, hipStream_t s);
void call_cache_give(void* p);
// hipMallocAsync; where memory is short, once more after every thread's unused blocks have gone back
hipError_t pool_alloc(void** p, size_t bytes, hipStream_t s);

struct Scratch {
    void* p = nullptr;
    hipStream_t s = nullptr;
    bool from_arena = false, from_cache = false;
    Scratch() = default;
    Scratch(const Scratch&) = delete;
    Scratch& operator=(const Scratch&) = delete;
    ~Scratch() { release(); }
    int alloc(size_t bytes, hipStream_t stream) {
        release();
        s = stream;
        if (bytes == 0) bytes = 256;
        if (Arena* a = thread_arena()) {
            if ((p = a->take(bytes)) != nullptr) {
                from_arena = true;
                return NSC_OK;
            }
        }
        if ((p = call_cache_take(bytes, stream)) != nullptr) {
            from_cache = true;
            return NSC_OK;
        }
        const hipError_t e = pool_alloc(&p, bytes, stream);
        if (e != hipSuccess) {
            p = nullptr;
            set_error("hipMallocAsync(%zu) failed: %s", bytes, hipGetErrorString(e));
            return NSC_ERR_NOMEM;
        }
        return NSC_OK;
    }
    void release() {
        if (p) {
            if (from_arena) {
                Arena* a = thread_arena();
                if (!a || !a->give(p)) { /* arena gone: nothing to return */ }
            } else if (from_cache) {
                call_cache_give(p);
            } else {
                (void)hipFreeAsync(p, s);
            }
        }
        p = nullptr;
        from_arena = from_cache = false;
    }
    template <typename T>
    T* as() const { return static_cast<T*>(p); }
};

}  // namespace nsc
