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
struct Launch { hipStream_t stream; int device; fx::ResidentEnd end; std::set<long> behind; bool ended; };      // behind: those whose events its stream waits for
std::mutex mu;
std::vector<Launch> launches;
std::map<int, long> last;                      // resident launch of a device
std::map<hipStream_t, std::set<long>> waits;   // of a stream
std::map<hipEvent_t, long> events;             // launch that carries the event, or that it stands behind
std::set<long> owed;                           // ends of calls of other kinds that the next resident launch has to wait for
std::set<hipStream_t> capturing;
std::atomic<int> bad{0}, made{0}, carried{0}, waited{0}, recorded{0};
std::atomic<bool> stop{false}, threaded{false};      // with threads, a call may end while a launch is on its way: the next one waits for it
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
            bool free = rand() % 3 == 0;
            for (long b : l.behind) free = free && launches[b].ended;
            if (!free) continue;
            l.ended = true;
            if (l.end.word) __atomic_store_n(l.end.word, l.end.ticket, __ATOMIC_RELEASE);
        }
    }
}
hipError_t launch(hipStream_t st, hipEvent_t end) {
    std::lock_guard<std::mutex> lk(mu);
    if (fail_next) { fail_next = false; return hipErrorLaunchFailure; }
    const long n = (long)launches.size();
    const std::set<long> behind = waits[st];
    if (capturing.count(st)) {
        if (end || end_of->word) wrong("a captured launch takes part in the order");
        return hipSuccess;
    }
    if (last.count(device)) {
        const long p = last[device];
        const bool one_stream = launches[p].stream == st && st != hipStreamPerThread;
        if (!one_stream && !launches[p].ended && !behind.count(p)) wrong("launch " + std::to_string(n) + " beside launch " + std::to_string(p));
    }
    for (long o : owed)
        if (!threaded && launches[o].stream != st && !launches[o].ended && !behind.count(o)) wrong("launch " + std::to_string(n) + " ahead of call " + std::to_string(o));
    owed.clear();
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
    for (long i = 0; i < (long)launches.size(); i++)
        if (launches[i].stream == st) events[e] = i;
    owed.insert(events[e]);
    recorded++;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t st, hipEvent_t e, unsigned) {
    named("hipStreamWaitEvent", st);
    std::lock_guard<std::mutex> lk(mu);
    if (!events.count(e)) wrong("a wait for an event that no launch carries");
    else waits[st].insert(events[e]);
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
// a call of kernels of other kinds: whether an event is left behind it
static bool ordinary(int stream) {
    mine = handle(stream);
    {
        std::lock_guard<std::mutex> lk(mu);
        if (!capturing.count(mine)) launches.push_back({mine, device, {nullptr, 0}, waits[mine], false});
    }
    const int before = recorded;
    if (fx::resident_works(mine) != hipSuccess) wrong("a call's end is refused");
    return recorded != before;
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
    for (int i = 0; i < 50 && !(carried && waited); i++)
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
    // calls of other kinds: their turn comes ahead of the next launch on another stream
    drain();
    std::this_thread::sleep_for(std::chrono::nanoseconds(fx::kWorkNs));
    if (ordinary(1) || ordinary(2)) wrong("an event where no resident launch was made");
    go(1);
    go(1);
    if (ordinary(1)) wrong("an event on the only stream with resident launches");
    if (!ordinary(2) || !ordinary(3) || !ordinary(0)) wrong("no event behind a call beside resident launches");
    go(1);
    go(1);
    ordinary(2);
    go(2);
    if (!ordinary(2) || !ordinary(1)) wrong("no event where two streams have resident launches");
    go(1);
    go(2);
    set_capturing(2, true);
    if (ordinary(2)) wrong("an event into a capture");
    set_capturing(2, false);
    for (int i = 0; i < 3 * fx::kWorks; i++) ordinary(100 + i);       // more streams than places: the oldest ones are given up
    {
        std::lock_guard<std::mutex> lk(mu);
        while (owed.size() > (size_t)fx::kWorks) owed.erase(owed.begin());
    }
    go(1);
    drain();
    const int made_before = made;
    size_t n = launches.size();
    threaded = true;
    std::vector<std::thread> threads;
    for (int k = 0; k < 4; k++)
        threads.emplace_back([k] {
            for (int i = 0; i < 500; i++) {
                go(k < 2 ? k : k == 2 ? -1 : 3 + i / 100 % 3);
                if (i % 7 == k) ordinary(k);
            }
        });
    for (auto& t : threads) t.join();
    drain();
    stop = true;
    dev.join();
    n = launches.size() - n;
    printf("%zu launches and calls, %d events carried, %d recorded, %d waits\n", launches.size(), carried.load(), recorded.load(), waited.load());
    if (n < 2280 || made_before != 4 + fx::kWorks || made != made_before) wrong("launches are missing, or too much was made");      // a word and an event for each of two devices, the calls' events
    return bad != 0;
}
