// The order of resident launches (csrc/resident.h) against runtime calls that only keep a record, and a thread that ends the launches
// of every stream in order: what is called on which stream, and whether a launch may find the one before it at work.
// Prints what is wrong; the exit status says whether something is.
#include <hip/hip_runtime_api.h>
extern "C" hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t, hipEvent_t, hipEvent_t, int);
#include "../flexllm_amd/csrc/resident.h"
#include <atomic>
#include <deque>
#include <map>
#include <set>
#include <stdio.h>
#include <stdlib.h>
#include <string>
#include <vector>

namespace {
struct Launch { hipStream_t stream; int device; fx::ResidentEnd end; long behind; bool ended; };      // behind: the launch whose event its stream waits for
std::mutex mu;
std::vector<Launch> launches;
std::map<int, long> last;                      // of a device
std::map<hipStream_t, long> waits;             // of a stream: the latest launch that it waits for
std::map<hipEvent_t, long> events;             // launch that carries the event
std::set<hipStream_t> capturing;
std::atomic<int> bad{0}, made{0}, carried{0}, waited{0};
std::atomic<bool> stop{false};
thread_local hipStream_t mine = nullptr;       // the caller's stream: no call may name another one
thread_local int device = 0;
thread_local fx::ResidentEnd* end_of = nullptr;
bool fail_next = false;

void wrong(const std::string& s) { printf("%s\n", s.c_str()); bad++; }
void named(const char* call, hipStream_t st) {
    if (st != mine) wrong(std::string(call) + " on another stream than the caller's");
}
// Ends launches as a device would: each behind those of its stream and the one that it waits for.
void run_device() {
    size_t from = 0;
    while (!stop) {
        std::this_thread::sleep_for(std::chrono::microseconds(50));
        std::lock_guard<std::mutex> lk(mu);
        while (from < launches.size() && launches[from].ended) from++;
        std::set<hipStream_t> busy;
        for (size_t i = from; i < launches.size(); i++) {
            Launch& l = launches[i];
            if (l.ended || busy.count(l.stream)) continue;
            busy.insert(l.stream);
            if ((l.behind >= 0 && !launches[l.behind].ended) || rand() % 3) continue;
            l.ended = true;
            if (l.end.word) __atomic_store_n(l.end.word, l.end.ticket, __ATOMIC_RELEASE);
        }
    }
}
hipError_t launch(hipStream_t st, hipEvent_t end) {
    std::lock_guard<std::mutex> lk(mu);
    if (fail_next) { fail_next = false; return hipErrorLaunchFailure; }
    const long n = (long)launches.size(), behind = waits.count(st) ? waits[st] : -1;
    if (capturing.count(st)) {
        if (end || end_of->word) wrong("a captured launch takes part in the order");
        return hipSuccess;
    }
    if (last.count(device)) {
        const long p = last[device];
        const bool one_stream = launches[p].stream == st && st != hipStreamPerThread;
        if (!one_stream && !launches[p].ended && behind < p) wrong("launch " + std::to_string(n) + " beside launch " + std::to_string(p));
    }
    launches.push_back({st, device, *end_of, behind, false});
    last[device] = n;
    if (end) { events[end] = n; carried++; }
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { made++; *p = calloc(n, 1); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus* s) {
    named("hipStreamIsCapturing", st);
    std::lock_guard<std::mutex> lk(mu);
    *s = capturing.count(st) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t st) { named("hipStreamQuery", st); return hipErrorNotReady; }
hipError_t hipStreamSynchronize(hipStream_t st) { named("hipStreamSynchronize", st); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)(uintptr_t)(0x1000 + 16 * ++made); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t st) {
    named("hipEventRecord", st);
    std::lock_guard<std::mutex> lk(mu);
    if (capturing.count(st)) wrong("an event joins a stream's capture");
    events[e] = last.count(device) ? last[device] : -1;
    carried++;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned) {
    named("hipStreamWaitEvent", st);
    std::lock_guard<std::mutex> lk(mu);
    if (!events.count(e)) wrong("a wait for an event that no launch carries");
    else if (!waits.count(st) || waits[st] < events[e]) waits[st] = events[e];
    waited++;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t st) { named("hipLaunchKernel", st); return launch(st, nullptr); }
hipError_t hipExtLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t st, hipEvent_t begin, hipEvent_t end, int) {
    named("hipExtLaunchKernel", st);
    if (begin) wrong("an event ahead of the launch");
    return launch(st, end);
}
}

static hipStream_t handle(int stream) { return stream < 0 ? hipStreamPerThread : (hipStream_t)(uintptr_t)(16 * stream); }      // 0: the null stream
static int go(int stream) {
    mine = handle(stream);
    fx::ResidentEnd end;
    end_of = &end;
    return (int)fx::resident_run(nullptr, 256, 512, nullptr, 0, mine, end);
}
static void set_capturing(int stream, bool on) {
    std::lock_guard<std::mutex> lk(mu);
    if (on) capturing.insert(handle(stream));
    else capturing.erase(handle(stream));
}
static void drain() {
    for (bool all = false; !all;) {
        std::this_thread::sleep_for(std::chrono::microseconds(200));
        std::lock_guard<std::mutex> lk(mu);
        all = true;
        for (auto& l : launches) all = all && l.ended;
    }
}

int main() {
    std::thread dev(run_device);
    // one stream, and several that never meet, whoever made them: no event
    for (int s : {5, 5, 5, 5}) go(s);
    for (int s : {1, 2, 0, 3, -1}) { drain(); go(s); }
    if (carried || waited) wrong("events without a meeting");
    for (int s : {1, 1, 2, 1, 0, 2, 2, 0, 3, -1, -1, 1}) go(s);
    if (!carried || !waited) wrong("no events where streams meet");
    // the last launch's stream begins a capture (a caller's own: the library does not hear of it), in and out of a meeting
    for (int k = 0; k < 2; k++) {
        go(1);
        set_capturing(1, true);
        go(2);
        go(1);                                            // into the capture
        go(3);
        set_capturing(1, false);
        go(1);
        for (int i = 0; i < fx::kSpell; i++) go(1);       // the events end
    }
    // a meeting that is over costs nothing any more
    drain();
    const int before = carried;
    for (int i = 0; i < 10; i++) go(1);
    if (carried != before) wrong("events long after a meeting");
    fail_next = true;
    if (go(1) != (int)hipErrorLaunchFailure) wrong("a failed launch is not reported");
    for (int s : {3, 1}) go(s);
    device = 1;
    go(4);
    device = 0;
    go(1);
    size_t n = launches.size();
    std::vector<std::thread> threads;
    for (int k = 0; k < 4; k++)
        threads.emplace_back([k] { for (int i = 0; i < 500; i++) go(k < 2 ? k : k == 2 ? -1 : 3 + i / 100 % 3); });
    for (auto& t : threads) t.join();
    drain();
    stop = true;
    dev.join();
    n = launches.size() - n;
    printf("%zu launches, %d events carried, %d waits\n", launches.size(), carried.load(), waited.load());
    if (n != 2000 || made != 4) wrong("launches are missing, or too much was made");      // a word and an event for each of two devices
    return bad != 0;
}
