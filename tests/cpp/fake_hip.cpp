// A HIP runtime without a device, preloaded over the real one by tests/test_host_dispatch.py: memory is the
// host's, streams and events are inert, launches run nothing and are counted by kernel name. It lets the
// library's host code (planning, scratch, dispatch) run on the CPU, with allocations that can be refused.
// fake_hip_limit(n) refuses every later hipMalloc of more than n bytes, leaving the error pending as the
// runtime does; fake_hip_launches() lists the kernels launched since the last call, one a line.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
size_t limit_bytes = ~size_t(0);
hipError_t pending = hipSuccess;
std::map<const void *, std::string> names;
std::string launched, listed;
char symbols[1 << 16];

hipError_t raise_error(hipError_t e) { return pending = e; }
void *handle() { return std::malloc(16); }
}  // namespace

extern "C" {

void fake_hip_limit(size_t n) { limit_bytes = n; }
const char *fake_hip_launches(void) {
    listed.swap(launched);
    launched.clear();
    return listed.c_str();
}

void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
    launched += names[f] + "\n";
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = symbols; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
const char *hipGetErrorName(hipError_t) { return "error"; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError(void) {
    const hipError_t e = pending;
    pending = hipSuccess;
    return e;
}

hipError_t hipMalloc(void **p, size_t n) {
    if (n > limit_bytes) return raise_error(hipErrorOutOfMemory);
    *p = std::aligned_alloc(256, (n + 255) / 256 * 256);
    return *p ? hipSuccess : raise_error(hipErrorOutOfMemory);
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memmove(d, s, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)handle(); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)handle(); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t)handle();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { std::free(g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t g) { std::free(g); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)handle(); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)handle(); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }

}  // extern "C"
