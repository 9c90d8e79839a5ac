// The HIP calls that the native library's host code makes, answered in host memory without a GPU: memory
// is malloc's, streams and events are tokens, kernels are not run.  A test loads it before the library
// (tests/test_host_paths.py), makes calls fail, and reads what was allocated and launched.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>

namespace {

struct Counts {
    long long device_allocs, device_bytes;  // bytes: held now
    long long host_allocs, host_bytes, host_peak;
    long long launches;
    unsigned long long workgroups;  // of the last launch
};
Counts counts;
std::map<void*, size_t> device, host;
hipError_t last = hipSuccess;
hipError_t fail_memcpy = hipSuccess, fail_launch = hipSuccess;
void** last_args = nullptr;  // of the running launch
unsigned char arg_copy[256];
int copy_arg = -1, copy_bytes = 0;
long long host_limit = 1ll << 40;

hipError_t done(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}

// What a launch may hold: the packet counts threads per dimension in 32 bits.
hipError_t launch(dim3 g, dim3 b, void** args) {
    if (fail_launch != hipSuccess) return done(fail_launch);
    if ((unsigned long long)b.x * b.y * b.z > 1024 || (unsigned long long)g.x * b.x > 0xffffffffull || g.y > 65535 || g.z > 65535)
        return done(hipErrorInvalidConfiguration);
    counts.launches++;
    counts.workgroups = (unsigned long long)g.x * g.y * g.z;
    if (copy_arg >= 0 && args) std::memcpy(arg_copy, args[copy_arg], (size_t)copy_bytes);
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- for the test
const Counts* host_hip_counts() { return &counts; }
void host_hip_fail(int memcpy_error, int launch_error) {
    fail_memcpy = (hipError_t)memcpy_error;
    fail_launch = (hipError_t)launch_error;
}
void host_hip_copy_arg(int arg, int bytes) {  // keep that argument of the launches that follow (-1: none)
    copy_arg = arg;
    copy_bytes = bytes;
}
void host_hip_limit(long long bytes) { host_limit = bytes; }  // of pinned host memory
const unsigned char* host_hip_arg() { return arg_copy; }
void host_hip_reset_peak() { counts.host_peak = counts.host_bytes; }

// ---- device and streams
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char symbol[256];
    *p = symbol;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free((void*)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free((void*)e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void** p, size_t n) {
    if (n > (size_t)1 << 40) return done(hipErrorOutOfMemory);
    *p = std::calloc(n ? n : 1, 1);
    device[*p] = n;
    counts.device_allocs++;
    counts.device_bytes += (long long)n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = device.find(p);
    if (it == device.end()) return done(p ? hipErrorInvalidValue : hipSuccess);
    counts.device_bytes -= (long long)it->second;
    device.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (counts.host_bytes + (long long)n > host_limit) return done(hipErrorOutOfMemory);
    *p = std::calloc(n ? n : 1, 1);
    host[*p] = n;
    counts.host_allocs++;
    counts.host_bytes += (long long)n;
    if (counts.host_bytes > counts.host_peak) counts.host_peak = counts.host_bytes;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    auto it = host.find(p);
    if (it == host.end()) return done(p ? hipErrorInvalidValue : hipSuccess);
    counts.host_bytes -= (long long)it->second;
    host.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* to, const void* from, size_t n, hipMemcpyKind) {
    if (fail_memcpy != hipSuccess) return done(fail_memcpy);
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* to, const void* from, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(to, from, n, k); }
hipError_t hipMemset(void* p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }

// ---- modules and launches
hipError_t hipModuleLoadData(hipModule_t* m, const void*) { *m = (hipModule_t)std::malloc(1); return hipSuccess; }
hipError_t hipModuleUnload(hipModule_t m) { std::free((void*)m); return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char*) { *f = (hipFunction_t)&counts; return hipSuccess; }
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz,
                                 unsigned, hipStream_t, void** args, void**) {
    return launch(dim3(gx, gy, gz), dim3(bx, by, bz), args);
}
hipError_t hipLaunchKernel(const void*, dim3 g, dim3 b, void** args, size_t, hipStream_t) {
    return launch(g, b, args);
}

}  // extern "C"
