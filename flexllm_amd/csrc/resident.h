// Order of the launches of kernels whose workgroups wait for each other and so have to be resident all at once.  Host code only,
// behind <hip/hip_ext.h> (which has no form for host compilers).
#pragma once
#include <hip/hip_runtime_api.h>
#include <atomic>
#include <chrono>
#include <mutex>
#include <thread>

namespace fx {

// Last parameter of such a kernel.  Its first workgroup, which ends behind words of all others, writes the launch's number at its end
// (resident_done): from then on all workgroups have been resident, and what is left of them ends by itself.  Null: nobody asks.
struct ResidentEnd {
    unsigned* word;                                       // host memory, one per device
    unsigned ticket;
};

// Two such kernels side by side could each hold a part of the chip and wait for the rest of it, so on a device they run one after the
// other, whatever streams and threads they are launched from (kernels of other kinds end by themselves).  No call made here names
// another stream than the caller's: that stream may be in the middle of a capture, or gone.
// Launches on one stream, or behind the last one's end, need nothing.  Where another stream's launch is still at work, the next one waits
// for the event that it carries; it carries one for kSpell launches behind such a meeting, since an event costs 4.2 us of the stream's
// time, and the word 0.2 (a short kernel and one of 100 us in turn; one step of Llama on a caller's stream 303.4 us with an event
// behind each, 297.6 so).  The first launch of such a meeting finds no event and holds its caller until the word is there, or for
// a minute: that stream may wait for something that this caller does next.
// In a stream that is being captured there is no order to keep: the launch runs when its graph does.
constexpr int kMaxDevices = 64, kSpell = 64;
constexpr long long kHoldNs = 60000000000;

// Calls of many kernels that end by themselves (prompts, steps of several tokens, sampled tokens), on other streams than the resident
// launches: between two of those one kernel gets in, so that a prompt of 150 kernels beside loops of 16 tokens takes a second.  Such a call
// leaves an event behind its last kernel, for which the next resident launch waits: they take turns.  16 layers of 2048, loops of 16
// tokens and prompts of 1531 on a stream each: 70 prompts and 1126 tokens a second, one prompt and 1663 tokens without that, 172 and
// 633 where the tokens come from a chain of kernels too.  Only where a resident launch on another stream was made in the last second.
constexpr int kWorks = 16;                                // streams with such calls; with more, the oldest one's is not waited for
constexpr long long kWorkNs = 1000000000;
struct ResidentWorks {
    std::mutex mu;
    struct { hipStream_t stream; hipEvent_t end; bool pending; unsigned long long age; } work[kWorks] = {};
    unsigned long long calls = 0;
    std::atomic<hipStream_t> where{nullptr};              // stream of the last resident launch,
    std::atomic<long long> when{-kWorkNs}, when_other{-kWorkNs};       // its time, and that of the last one on any other stream
};
inline long long resident_clock() { return std::chrono::duration_cast<std::chrono::nanoseconds>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

struct ResidentTurn {
    ResidentWorks works;
    std::mutex mu;                                        // launches have one order
    unsigned* word = nullptr;
    hipEvent_t end = nullptr;                             // of the last launch, where it carries one
    hipStream_t last = nullptr;
    unsigned ticket = 0;                                  // of the last launch
    bool carries = false;
    int spell = 0;                                        // further launches that carry events
    hipError_t prepare() {
        hipError_t e = hipSuccess;
        if (!end) e = hipEventCreateWithFlags(&end, hipEventDisableTiming);
        if (e == hipSuccess && !word) {
            void* p = nullptr;
            e = hipHostMalloc(&p, 64, hipHostMallocPortable);
            if (e == hipSuccess) {
                word = static_cast<unsigned*>(p);
                *word = 0;
            }
        }
        return e;
    }
    bool done() const { return __atomic_load_n(word, __ATOMIC_ACQUIRE) == ticket; }
};
inline hipError_t resident_turn(ResidentTurn*& t) {       // of the current device
    static ResidentTurn turns[kMaxDevices];
    int dev = 0;
    const hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess && (dev < 0 || dev >= kMaxDevices)) return hipErrorInvalidDevice;
    t = &turns[dev];
    return e;
}
// What launches need besides, so that none of them allocates.
inline hipError_t resident_prepare() {
    ResidentTurn* t = nullptr;
    const hipError_t e = resident_turn(t);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(t->mu);
    return t->prepare();
}
// end: the last of the kernel's arguments, set here.
inline hipError_t resident_run(const void* kernel, int grid, int block, void** args, size_t lds, hipStream_t st, ResidentEnd& end) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &cap);
    if (e != hipSuccess) return e;
    end = {nullptr, 0};
    if (cap != hipStreamCaptureStatusNone) return hipLaunchKernel(kernel, dim3(grid), dim3(block), args, lds, st);
    ResidentTurn* t = nullptr;
    e = resident_turn(t);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lk(t->mu);
    e = t->prepare();
    if (e != hipSuccess) return e;
    // hipStreamPerThread is another stream in every thread
    if ((st != t->last || st == hipStreamPerThread) && !t->done()) {
        if (t->carries) e = hipStreamWaitEvent(st, t->end, 0);
        else for (const long long until = resident_clock() + kHoldNs; !t->done() && resident_clock() < until;) std::this_thread::sleep_for(std::chrono::microseconds(20));
        if (e != hipSuccess) return e;
        t->spell = kSpell;
    }
    {
        std::lock_guard<std::mutex> works(t->works.mu);
        for (auto& w : t->works.work) {
            if (!w.pending) continue;
            if (w.stream != st || st == hipStreamPerThread) e = hipStreamWaitEvent(st, w.end, 0);
            if (e != hipSuccess) return e;
            w.pending = false;                            // later launches come behind this one
        }
        if (t->works.where.load(std::memory_order_relaxed) != st) {
            t->works.when_other.store(t->works.when.load(std::memory_order_relaxed), std::memory_order_relaxed);
            t->works.where.store(st, std::memory_order_relaxed);
        }
        t->works.when.store(resident_clock(), std::memory_order_relaxed);
    }
    end = {t->word, t->ticket + 1};
    const bool carries = t->spell > 0;
    e = carries ? hipExtLaunchKernel(kernel, dim3(grid), dim3(block), args, lds, st, nullptr, t->end, 0)
                : hipLaunchKernel(kernel, dim3(grid), dim3(block), args, lds, st);
    if (e != hipSuccess) return e;
    t->last = st;
    t->ticket++;
    t->carries = carries;
    t->spell -= carries;
    return e;
}
// Behind the last kernel of a call as described above.
inline hipError_t resident_works(hipStream_t st) {
    ResidentTurn* t = nullptr;
    hipError_t e = resident_turn(t);
    if (e != hipSuccess) return e;
    ResidentWorks& all = t->works;
    const bool own = all.where.load(std::memory_order_relaxed) == st && st != hipStreamPerThread;
    if (resident_clock() - (own ? all.when_other : all.when).load(std::memory_order_relaxed) >= kWorkNs) return hipSuccess;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    e = hipStreamIsCapturing(st, &cap);
    if (e != hipSuccess || cap != hipStreamCaptureStatusNone) return e;
    std::lock_guard<std::mutex> lk(all.mu);
    auto* w = &all.work[0];
    for (auto& x : all.work) {                            // the stream's own place, a free one, or the oldest
        if (x.end && x.stream == st) { w = &x; break; }
        if (x.age < w->age) w = &x;
    }
    if (!w->end) e = hipEventCreateWithFlags(&w->end, hipEventDisableTiming | hipEventDisableSystemFence);
    if (e == hipSuccess) e = hipEventRecord(w->end, st);
    if (e != hipSuccess) return e;
    w->stream = st;
    w->pending = true;
    w->age = ++all.calls;
    return e;
}

}  // namespace fx
