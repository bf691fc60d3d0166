// The call cache (nscale_amd/csrc/call_cache.cpp) against a stand-in for the HIP runtime: memory with a limit,
// streams and events whose work is done when the test says so, and the rule that a call which is unsafe while
// a stream is captured in global mode ends the capture.  Argument: the check to run.
#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "scratch.hpp"

namespace {
std::recursive_mutex mu;
struct Fake {
    std::map<void*, size_t> mem;
    size_t used = 0, limit = ~(size_t)0;
    size_t held = 0;       // freed bytes that the pool keeps until it is trimmed (with keeps)
    bool keeps = false;
    bool capturing = false, invalidated = false;  // some stream is being captured, in global mode
    struct Event { bool recorded = false, done = true; uintptr_t stream = 0; };
    std::vector<Event> events;
    std::map<uintptr_t, bool> busy;               // streams with work that has not ended
    std::vector<std::pair<uintptr_t, size_t>> waits;
    std::vector<uintptr_t> freed_on;
    int bad_frees = 0, own_streams = 0;
} F;
thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;
void unsafe() {
    if (F.capturing && mode != hipStreamCaptureModeRelaxed) F.invalidated = true;
}
typedef std::lock_guard<std::recursive_mutex> Lock;
int failures = 0;
#define EXPECT(c) do { if (!(c)) { ++failures; std::printf("line %d: %s\n", __LINE__, #c); } } while (0)
hipStream_t stream(uintptr_t n) { return reinterpret_cast<hipStream_t>(n * 64); }
}  // namespace

namespace nsc {
void set_error(const char*, ...) {}
Arena*& thread_arena() { static thread_local Arena* a = nullptr; return a; }
}  // namespace nsc

extern "C" {
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) {
    Lock l(mu);
    if (F.used + F.held + n > F.limit) return hipErrorOutOfMemory;
    *p = std::malloc(1);
    F.mem[*p] = n;
    F.used += n;
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t s) {
    Lock l(mu);
    if (!s && F.capturing) F.invalidated = true;  // the legacy stream waits for the captured one
    auto it = F.mem.find(p);
    if (it == F.mem.end()) { ++F.bad_frees; return hipErrorInvalidValue; }
    F.used -= it->second;
    if (F.keeps) F.held += it->second;
    F.freed_on.push_back(reinterpret_cast<uintptr_t>(s));
    F.mem.erase(it);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    Lock l(mu);
    F.events.emplace_back();
    *e = reinterpret_cast<hipEvent_t>(F.events.size());
    return hipSuccess;
}
static Fake::Event& ev(hipEvent_t e) { return F.events[reinterpret_cast<size_t>(e) - 1]; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Lock l(mu);
    ev(e).recorded = true;
    ev(e).stream = reinterpret_cast<uintptr_t>(s);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    Lock l(mu);
    unsafe();
    return F.busy[ev(e).stream] ? hipErrorNotReady : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    Lock l(mu);
    unsafe();
    F.busy[ev(e).stream] = false;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    Lock l(mu);
    F.waits.emplace_back(reinterpret_cast<uintptr_t>(s), ev(e).stream);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    Lock l(mu);
    *st = hipStreamCaptureStatusNone;
    return !s && F.capturing ? hipErrorStreamCaptureImplicit : hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    std::swap(*m, mode);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    Lock l(mu);
    *s = stream(1000 + ++F.own_streams);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    Lock l(mu);
    unsafe();
    F.busy[reinterpret_cast<uintptr_t>(s)] = false;
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t* p, int) { *p = nullptr; return hipSuccess; }
hipError_t hipMemPoolTrimTo(hipMemPool_t, size_t) { Lock l(mu); F.held = 0; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace {
constexpr size_t MB = (size_t)1 << 20;
// one operator call with one buffer; its work stays on the stream until end_work
int call(uintptr_t s, size_t bytes) {
    nsc::Scratch sc;
    const int rc = sc.alloc(bytes, stream(s));
    Lock l(mu);
    F.busy[reinterpret_cast<uintptr_t>(stream(s))] = true;
    return rc;
}
void end_work() { Lock l(mu); F.busy.clear(); }

// calls on other streams, and the end of a thread that made some, leave a global capture alone
void capture() {
    for (uintptr_t s = 1; s <= 3; ++s) EXPECT(call(s, 3 * MB) == NSC_OK);
    std::thread t([] {
        EXPECT(call(7, MB) == NSC_OK);
        F.capturing = true;
        for (uintptr_t s = 1; s <= 7; ++s) EXPECT(call(s, 2 * MB) == NSC_OK);
    });
    t.join();
    for (uintptr_t s = 1; s <= 6; ++s) EXPECT(call(s, 2 * MB) == NSC_OK);
    EXPECT(!F.invalidated);
    EXPECT(mode == hipStreamCaptureModeGlobal);
    F.capturing = false;
}

// an allocation that fails finds the memory of unused blocks: this thread's and other threads', with work
// that has ended and with work that the stream has to wait for, with a pool that reuses and one that keeps
void pressure() {
    for (bool keeps : {false, true}) {
        F.keeps = keeps;
        F.limit = ~(size_t)0;
        for (uintptr_t s = 1; s <= 3; ++s) EXPECT(call(s, 900 * MB) == NSC_OK);
        EXPECT(F.used > 2700 * MB);
        F.limit = 3400 * MB;
        F.waits.clear();
        F.freed_on.clear();
        EXPECT(call(4, 2500 * MB) == NSC_OK);  // above a block's bound: the pool's own
        EXPECT(F.waits.size() == 3 && F.freed_on.size() == 4);  // three blocks, then the buffer itself
        for (auto& w : F.waits) EXPECT(w.first == reinterpret_cast<uintptr_t>(stream(4)));
        for (uintptr_t q : F.freed_on) EXPECT(q == reinterpret_cast<uintptr_t>(stream(4)));
        end_work();
        F.held = 0;
    }
    F.keeps = false;
    // another thread's blocks, while it lives and makes no call
    std::mutex gate;
    gate.lock();
    std::atomic<bool> ready{false};
    std::thread other([&] {
        EXPECT(call(8, 900 * MB) == NSC_OK);
        EXPECT(call(9, 900 * MB) == NSC_OK);
        ready = true;
        gate.lock();
        EXPECT(call(8, 100 * MB) == NSC_OK);  // and goes on without them
        gate.unlock();
    });
    while (!ready) std::this_thread::yield();
    F.limit = 3000 * MB;
    EXPECT(call(4, 2500 * MB) == NSC_OK);
    gate.unlock();
    other.join();
    // a block that a call holds is kept, and the failure is reported
    {
        nsc::Scratch a, b;
        EXPECT(a.alloc(500 * MB, stream(1)) == NSC_OK);
        const size_t before = F.used;
        EXPECT(b.alloc(2900 * MB, stream(1)) == NSC_ERR_NOMEM);
        EXPECT(F.used == before && F.mem.size() == 1);
    }
    // nothing is given back on a captured stream's behalf, and the capture goes on
    F.capturing = true;
    EXPECT(call(0, 2900 * MB) == NSC_ERR_NOMEM);
    EXPECT(!F.invalidated);
    F.capturing = false;
}

// blocks of streams that have gone quiet go back while the thread works on another one
void age() {
    for (uintptr_t s = 1; s <= 4; ++s) EXPECT(call(s, 300 * MB) == NSC_OK);
    EXPECT(F.used >= 1200 * MB);
    end_work();
    for (int k = 0; k < 200; ++k) EXPECT(call(1, 300 * MB) == NSC_OK);
    EXPECT(F.used >= 300 * MB && F.used < 400 * MB);
    for (uintptr_t s = 2; s <= 4; ++s) EXPECT(call(s, 300 * MB) == NSC_OK);
    EXPECT(F.used >= 1200 * MB);
    // streams in turn: none of them is quiet
    const size_t before = F.used;
    for (int k = 0; k < 800; ++k) EXPECT(call(1 + k % 4, 300 * MB) == NSC_OK);
    EXPECT(F.used == before);
}
}  // namespace

int main(int argc, char** argv) {
    const char* what = argc > 1 ? argv[1] : "";
    std::thread t([&] {  // its end gives its blocks back
        if (!std::strcmp(what, "capture")) capture();
        else if (!std::strcmp(what, "pressure")) pressure();
        else if (!std::strcmp(what, "age")) age();
        else EXPECT(!"a check of that name");
    });
    t.join();
    F.limit = ~(size_t)0;
    EXPECT(F.mem.empty() && F.used == 0 && !F.bad_frees);
    if (failures) std::printf("%s: %d failures\n", what, failures);
    return failures != 0;
}
