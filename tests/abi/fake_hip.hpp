// A HIP runtime without a GPU, for host programs linked against libdghip.so: the program's definitions take the place of
// libamdhip64's.  Device memory is host memory, copies are done at once, kernels are noted and not run.  Allocations and
// launches can be made to fail, and the queued work of every stream is followed through events and waits, so that a test
// can ask what may still be running.  Include it in one source file of a program.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <vector>

namespace fake {

struct Stream;
typedef std::map<Stream*, long> Waits;   // work of streams, as the number of launches it reaches to
struct Stream {
    long issued = 0, done = 0;   // launches queued here, and known to have ended
    Waits waits;                 // what later work here waits for
};
struct Event {
    Waits waits;
};
inline void add(Waits& w, Stream* s, long at) {
    long& x = w[s];
    if (x < at) x = at;
}

struct State {
    std::recursive_mutex mu;
    std::map<const void*, std::string> kernels;      // by host stub: the mangled name
    std::set<Stream*> streams;
    std::map<void*, size_t> device, pinned;          // live allocations
    int mallocs = 0, fail_malloc = 0;                // the fail_malloc-th hipMalloc from now on fails (0: none)
    int launches = 0, fail_launch = 0;
    size_t pinned_bytes = 0;
    hipError_t last = hipSuccess;
    std::function<void(const std::string&, void**)> on_launch;
    std::function<void(void* dst, const void* src, size_t n, hipMemcpyKind)> on_copy;   // called without the lock
    std::function<void()> on_sync;
};
inline State& state() {
    static State* s = new State;   // the library registers its kernels before this program's initialisers run
    return *s;
}
inline void finish(const Waits& waits) {
    for (auto& w : waits)
        if (w.first->done < w.second) w.first->done = w.second;
}
// launches that no synchronisation has waited for
inline long pending() {
    std::lock_guard<std::recursive_mutex> lock(state().mu);
    long n = 0;
    for (Stream* s : state().streams) n += s->issued - s->done;
    return n;
}

}  // namespace fake

#define FAKE_LOCK std::lock_guard<std::recursive_mutex> lock(fake::state().mu)
static fake::Stream* fs(hipStream_t s) { return reinterpret_cast<fake::Stream*>(s); }
static fake::Event* fe(hipEvent_t e) { return reinterpret_cast<fake::Event*>(e); }

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    fake::state().kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static thread_local struct { dim3 g, b; size_t m; hipStream_t s; } pushed;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) {
    pushed = {g, b, m, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s) {
    *g = pushed.g; *b = pushed.b; *m = pushed.m; *s = pushed.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t s) {
    FAKE_LOCK;
    fake::State& st = fake::state();
    ++st.launches;
    if (st.fail_launch && --st.fail_launch == 0) return st.last = hipErrorLaunchFailure;
    ++fs(s)->issued;
    if (st.on_launch) st.on_launch(st.kernels[f], args);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    FAKE_LOCK;
    const hipError_t e = fake::state().last;
    fake::state().last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {   // the header names the current version of it
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char scratch[1 << 16];
    *p = scratch;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 1; return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
    FAKE_LOCK;
    fake::State& st = fake::state();
    ++st.mallocs;
    *p = nullptr;
    if (st.fail_malloc && --st.fail_malloc == 0) return st.last = hipErrorOutOfMemory;
    *p = std::calloc(1, n ? n : 1);
    st.device[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    FAKE_LOCK;
    if (p && !fake::state().device.erase(p)) std::abort();   // freed twice, or never allocated
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    FAKE_LOCK;
    *p = std::calloc(1, n);
    fake::state().pinned[*p] = n;
    fake::state().pinned_bytes += n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    FAKE_LOCK;
    auto it = fake::state().pinned.find(p);
    if (it == fake::state().pinned.end()) std::abort();
    fake::state().pinned_bytes -= it->second;
    fake::state().pinned.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
    std::memcpy(d, s, n);
    if (fake::state().on_copy) fake::state().on_copy(d, s, n, k);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    FAKE_LOCK;
    auto* p = new fake::Stream;
    fake::state().streams.insert(p);
    *s = reinterpret_cast<hipStream_t>(p);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }   // kept: events may name it
hipError_t hipStreamSynchronize(hipStream_t s) {
    {
        FAKE_LOCK;
        fs(s)->done = fs(s)->issued;
        fake::finish(fs(s)->waits);
    }
    if (fake::state().on_sync) fake::state().on_sync();
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    FAKE_LOCK;
    for (auto& w : fe(e)->waits) fake::add(fs(s)->waits, w.first, w.second);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new fake::Event);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete fe(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    FAKE_LOCK;
    fe(e)->waits = fs(s)->waits;
    fake::add(fe(e)->waits, fs(s), fs(s)->issued);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    FAKE_LOCK;
    fake::finish(fe(e)->waits);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { *x = nullptr; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
