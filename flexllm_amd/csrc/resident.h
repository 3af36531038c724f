// Order of the launches of kernels whose workgroups wait for each other and so have to be resident all at once.  Host code only,
// behind <hip/hip_ext.h> (which has no form for host compilers).
#pragma once
#include <hip/hip_runtime_api.h>
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
// behind each, 297.6 so).  The first launch of such a meeting finds no event and holds its caller until the word is there.
// In a stream that is being captured there is no order to keep: the launch runs when its graph does.
constexpr int kMaxDevices = 64, kSpell = 64;
struct ResidentTurn {
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
        else while (!t->done()) std::this_thread::sleep_for(std::chrono::microseconds(20));
        if (e != hipSuccess) return e;
        t->spell = kSpell;
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

}  // namespace fx
