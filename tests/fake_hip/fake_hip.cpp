// A HIP runtime that runs nothing and writes down what it is asked for, so
// that the host side of the library's step calls can be checked on a CPU:
// what is launched, captured, replayed and waited for, in which order and by
// which thread.  Loaded (RTLD_GLOBAL) before libmgad.so, whose calls it takes.
//
// Events of the log, one per call: L a kernel launched, C a copy, W the stream
// waited for, D the device; [ and ] the bounds of a capture, with n for a
// launch and c for a copy recorded in between (x for a launch or copy of
// another thread than the capturing one), Rk; a replay of a graph of k nodes.
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>

namespace {

struct Capture {
    std::thread::id by;
    long nodes = 0;
};
std::mutex m;
std::map<hipStream_t, Capture> captures;
std::string events;
int hold_ms = 0;
int live_execs = 0;
long last_groups = 0;

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config config;

hipError_t work(hipStream_t s, char direct, char recorded) {
    std::lock_guard<std::mutex> lock(m);
    const auto it = captures.find(s);
    if (it == captures.end()) {
        events += direct;
    } else {
        it->second.nodes++;
        events += it->second.by == std::this_thread::get_id() ? recorded : 'x';
    }
    return hipSuccess;
}

hipError_t note(char c) {
    std::lock_guard<std::mutex> lock(m);
    events += c;
    return hipSuccess;
}

}  // namespace

extern "C" {

// The log so far, cleared (the caller frees it).
char *fake_take_log() {
    std::lock_guard<std::mutex> lock(m);
    char *r = strdup(events.c_str());
    events.clear();
    return r;
}
// Every capture from now on stays open at least this long.
void fake_hold_captures(int ms) { hold_ms = ms; }
int fake_captures_open() {
    std::lock_guard<std::mutex> lock(m);
    return static_cast<int>(captures.size());
}
// Workgroups of the last launch.
long fake_last_groups() { return last_groups; }
int fake_live_execs() {
    std::lock_guard<std::mutex> lock(m);
    return live_execs;
}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    config = Config{grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 g, dim3, void **, size_t, hipStream_t s) {
    last_groups = 1l * g.x * g.y * g.z;
    return work(s, 'L', 'n');
}
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t s) { return work(s, 'C', 'c'); }
hipError_t hipStreamSynchronize(hipStream_t) { return note('W'); }
hipError_t hipDeviceSynchronize() { return note('D'); }

hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) {
    {
        std::lock_guard<std::mutex> lock(m);
        if (captures.count(s)) return hipErrorIllegalState;
        captures[s].by = std::this_thread::get_id();
        events += '[';
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(hold_ms));
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) {
    std::lock_guard<std::mutex> lock(m);
    const auto it = captures.find(s);
    if (it == captures.end()) return hipErrorIllegalState;
    *g = reinterpret_cast<hipGraph_t>(new long(it->second.nodes));
    captures.erase(it);
    events += ']';
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    std::lock_guard<std::mutex> lock(m);
    *st = captures.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t g, hipGraphNode_t *, char *, size_t) {
    std::lock_guard<std::mutex> lock(m);
    live_execs++;
    *e = reinterpret_cast<hipGraphExec_t>(new long(*reinterpret_cast<long *>(g)));
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    std::lock_guard<std::mutex> lock(m);
    events += "R" + std::to_string(*reinterpret_cast<long *>(e)) + ";";
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete reinterpret_cast<long *>(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    std::lock_guard<std::mutex> lock(m);
    live_execs--;
    delete reinterpret_cast<long *>(e);
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n) { return (*p = malloc(n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    return *n = 2, hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake"; }

}  // extern "C"
