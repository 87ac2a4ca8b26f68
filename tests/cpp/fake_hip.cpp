// A HIP runtime without a device, for CPU tests of the host side: loaded before the
// library, its functions take the place of the real ones.  Device memory is host memory
// (zeroed, and not returned to malloc before the end, so that an address names one
// allocation), kernels do nothing, and a captured graph is the list of its launches.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <dlfcn.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

struct Block {
    size_t bytes;
    int dev;
};
struct Launch {
    std::string kernel;
    std::vector<void*> ptr;
};
using Launches = std::vector<Launch>;

std::recursive_mutex mu;
std::map<char*, Block> live;
std::map<const void*, std::string>& kernels() {   // (needed before this file's globals are there)
    static auto* const m = new std::map<const void*, std::string>;
    return *m;
}
Launches* capturing = nullptr;
int device = 0;
long device_total = 0;          // bytes that may be allocated (0: no limit)
long used = 0;
long fail_after = -1;           // allocations from now on that still succeed (-1: all)
long stale = 0;                 // pointers of a replayed launch that are not allocated
std::string trace;              // frees and waits, in order

bool allocated(void* p) {
    auto it = live.upper_bound(static_cast<char*>(p));
    if (it == live.begin()) return false;
    --it;
    return static_cast<char*>(p) < it->first + it->second.bytes;
}

// leading arguments that are pointers, of the kernels whose launches a graph is checked for
int pointer_args(const std::string& name) {
    return name.find("ms_expand_kernel") != std::string::npos ? 16 : name.find("ms_side_kernel") != std::string::npos ? 7 : 0;
}

hipError_t launch(const void* f, void** args) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    if (!capturing) return hipSuccess;
    Launch l{kernels()[f], {}};
    for (int i = 0; i < pointer_args(l.kernel); i++) l.ptr.push_back(*static_cast<void**>(args[i]));
    capturing->push_back(l);
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- for the test
void fake_fail_after(long n) { fail_after = n; }
void fake_device_total(long bytes) { device_total = bytes; }
long fake_used() { return used; }
long fake_stale() { return stale; }
const char* fake_trace() { return trace.c_str(); }
void fake_clear_trace() { trace.clear(); }

// ---- the runtime
void __hipRegisterFunction(void** modules, const void* host, char* dev, const char* name, unsigned limit, void* tid,
                           void* bid, void* block, void* grid, int* size) {
    kernels()[host] = name;
    using F = void (*)(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*);
    static const F real = reinterpret_cast<F>(dlsym(RTLD_NEXT, "__hipRegisterFunction"));
    if (real) real(modules, host, dev, name, limit, tid, bid, block, grid, size);
}

hipError_t hipMalloc(void** p, size_t bytes) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    *p = nullptr;
    if (fail_after == 0 || (device_total > 0 && used + (long)bytes > device_total)) return hipErrorOutOfMemory;
    if (fail_after > 0) fail_after--;
    *p = std::calloc(1, bytes);
    live[static_cast<char*>(*p)] = Block{bytes, device};
    used += (long)bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    const auto it = live.find(static_cast<char*>(p));
    if (it == live.end()) return p ? hipErrorInvalidValue : hipSuccess;
    trace += "free@" + std::to_string(it->second.dev) + " ";
    used -= (long)it->second.bytes;
    live.erase(it);   // (the memory stays: see above)
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* fr, size_t* total) {
    *total = device_total > 0 ? (size_t)device_total : (size_t)1 << 36;
    *fr = *total - (size_t)used;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return (*p = std::calloc(1, bytes)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void*) { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }

hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
hipError_t hipSetDevice(int d) { return device = d, hipSuccess; }
hipError_t hipDeviceSynchronize() {
    std::lock_guard<std::recursive_mutex> lock(mu);
    trace += "wait@" + std::to_string(device) + " ";
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipFuncGetAttributes(hipFuncAttributes*, const void*) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = reinterpret_cast<hipStream_t>(std::calloc(1, 16)), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = reinterpret_cast<hipEvent_t>(std::calloc(1, 16)), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
    *grid = *block = dim3(1);
    *lds = 0;
    *st = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) { return launch(f, args); }
hipError_t hipExtLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) {
    return launch(f, args);
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return capturing = new Launches, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    *g = reinterpret_cast<hipGraph_t>(capturing);
    capturing = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
    return *x = reinterpret_cast<hipGraphExec_t>(g), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return delete reinterpret_cast<Launches*>(x), hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lock(mu);
    for (const Launch& l : *reinterpret_cast<Launches*>(x))
        for (void* p : l.ptr) stale += p && !allocated(p);
    return hipSuccess;
}

}  // extern "C"
