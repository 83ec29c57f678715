// A HIP runtime of the CPU for tests of the library's host code: two devices, streams, events, captures and memory that
// only remember what belongs to what.  Linked with the objects of the library under test in the place of libamdhip64; a
// kernel launched through it runs at once, as the host function registered for it here, or does nothing.
#pragma once
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <utility>
#include <vector>

namespace fake {

struct Stream {
    int device;
    bool capturing = false;
};
struct Event {
    int device;
};
struct Op {  // what reached a stream, in order
    std::string what;
    hipStream_t stream;
    std::thread::id thread;
    void* event;
};
struct State {
    std::mutex mutex;
    std::vector<Op> ops;
    std::map<const void*, std::string> kernels;  // host handle -> device name
    std::map<void*, int> memory;                 // allocation -> device, -1: pinned
    bool per_thread_capturing = false;
    unsigned busy_ms = 0;  // how long the GPU works before the next event is reached
    int errors = 0;  // calls a real runtime would have refused
};
inline State& state() {
    static State s;
    return s;
}
inline thread_local int current_device = 0;
struct Var {
    size_t bytes;
    std::map<int, std::vector<char>> by_device;
};
inline std::map<const void*, Var>& vars() {
    static std::map<const void*, Var> v;
    return v;
}
// what a test makes of a launch (the kernel's mangled name, its arguments)
inline std::function<void(const std::string&, dim3, void**, hipStream_t)>& on_launch() {
    static std::function<void(const std::string&, dim3, void**, hipStream_t)> f;
    return f;
}
inline thread_local dim3 push_grid, push_block;
inline thread_local int inside = 0;  // the runtime's own allocations are none of the library's
struct Inside {
    Inside() { inside++; }
    ~Inside() { inside--; }
};

inline void log(const char* what, hipStream_t stream, void* event = nullptr) {
    Inside here;
    std::lock_guard<std::mutex> lock(state().mutex);
    state().ops.push_back({what, stream, std::this_thread::get_id(), event});
}
inline bool is_handle(hipStream_t s) { return s == nullptr || s == hipStreamLegacy || s == hipStreamPerThread; }
inline int device_of(hipStream_t s) { return is_handle(s) ? current_device : ((Stream*)s)->device; }
inline hipError_t refuse(hipError_t e) {
    state().errors++;
    return e;
}

}  // namespace fake

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = fake::current_device, hipSuccess; }
hipError_t hipSetDevice(int d) { return fake::current_device = d, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    fake::Inside here;
    std::lock_guard<std::mutex> lock(fake::state().mutex);
    fake::state().memory[*p] = fake::current_device;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    fake::Inside here;
    std::lock_guard<std::mutex> lock(fake::state().mutex);
    fake::state().memory[*p] = -1;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    {
        std::lock_guard<std::mutex> lock(fake::state().mutex);
        if (!fake::state().memory.erase(p)) fake::state().errors++;
    }
    free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(d, s, n), hipSuccess; }

hipError_t hipStreamCreate(hipStream_t* s) { fake::Inside here; return *s = (hipStream_t) new fake::Stream{fake::current_device}, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete (fake::Stream*)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return fake::log("synchronize", s), hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* c) {
    const bool on = s == hipStreamPerThread ? fake::state().per_thread_capturing : !fake::is_handle(s) && ((fake::Stream*)s)->capturing;
    return *c = on ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode*) { return hipSuccess; }

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { fake::Inside here; return *e = (hipEvent_t) new fake::Event{fake::current_device}, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete (fake::Event*)e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (((fake::Event*)e)->device != fake::device_of(s)) return fake::refuse(hipErrorInvalidHandle);
    return fake::log("record", s, e), hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) {
    std::this_thread::sleep_for(std::chrono::milliseconds(std::exchange(fake::state().busy_ms, 0u)));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    hipStreamCaptureStatus c;
    (void)hipStreamIsCapturing(s, &c);
    if (c != hipStreamCaptureStatusNone) return fake::refuse(hipErrorStreamCaptureIsolation);
    return fake::log("wait", s, e), hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    fake::Inside here;
    std::lock_guard<std::mutex> lock(fake::state().mutex);
    auto it = fake::vars().find(symbol);
    if (it == fake::vars().end()) return hipErrorInvalidSymbol;
    auto& mem = it->second.by_device[fake::current_device];
    mem.resize(it->second.bytes + 256);
    *p = (void*)(((uintptr_t)mem.data() + 255) & ~(uintptr_t)255);
    return hipSuccess;
}

// what a compiled kernel launch calls
static void* fake_fatbin;
void** __hipRegisterFatBinary(const void*) { return &fake_fatbin; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    fake::state().kernels[host] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t bytes, int, int) { fake::vars()[var].bytes = bytes; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t s);
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* n, hipStream_t* s);
static thread_local hipStream_t fake_push_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t s) {
    fake::push_grid = g;
    fake::push_block = b;
    fake_push_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* n, hipStream_t* s) {
    *g = fake::push_grid;
    *b = fake::push_block;
    *n = 0;
    *s = fake_push_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3, void** args, size_t, hipStream_t s) {
    fake::Inside here;
    const std::string& name = fake::state().kernels[host];
    if (fake::on_launch()) fake::on_launch()(name, grid, args, s);
    if (name.find("stage_copy") != std::string::npos)
        memcpy(*(void**)args[0], *(void**)args[1], *(size_t*)args[2] * 16);
    return hipSuccess;
}
}
