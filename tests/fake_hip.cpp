// A HIP runtime without a device, for CPU tests of the host library's own
// decisions (routes, scratch, what a refused allocation leaves behind):
// allocations are host memory under a limit that the test sets, copies run,
// kernels do nothing.  Linked with zlm_gpu_hip.cpp into a library of its own.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <unordered_map>

namespace {
std::unordered_map<void*, size_t> live;  // device allocations
uint64_t live_bytes = 0, limit_bytes = UINT64_MAX;
uint64_t stats[7] = {};  // see fake_hip_stat
bool capturing = false;
char handle;
template <class T>
T a_handle() {
    return reinterpret_cast<T>(&handle);
}
}  // namespace

// 0 live device bytes, 1 allocations, 2 refused allocations, 3 frees, 4 stream
// synchronisations, 5 copies host to device, 6 copies device to host, 7 calls that
// a real runtime would not take (frees of what is not allocated, waits for a
// capturing stream).
enum { kMallocs, kRefused, kFrees, kSyncs, kH2d, kD2h, kMisuse };
extern "C" uint64_t fake_hip_stat(int i) { return i == 0 ? live_bytes : stats[i - 1]; }
extern "C" void fake_hip_limit(uint64_t bytes) { limit_bytes = bytes; }

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    memset(p, 0, sizeof *p);
    snprintf(p->name, sizeof p->name, "none");
    snprintf(p->gcnArchName, sizeof p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "refused"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t n) {
    if (live_bytes + n > limit_bytes) return stats[kRefused]++, *p = nullptr, hipErrorOutOfMemory;
    *p = calloc(1, n ? n : 1);
    live[*p] = n;
    live_bytes += n;
    return stats[kMallocs]++, hipSuccess;
}
hipError_t hipFree(void* p) {
    auto it = live.find(p);
    if (it == live.end()) return stats[kMisuse]++, hipErrorInvalidValue;
    live_bytes -= it->second;
    live.erase(it);
    free(p);
    return stats[kFrees]++, hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = calloc(1, n ? n : 1), hipSuccess; }
hipError_t hipHostFree(void* p) { return free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { return *f = *t = 1 << 30, hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind kind) {
    memcpy(d, s, n);
    if (kind == hipMemcpyHostToDevice) stats[kH2d]++;
    if (kind == hipMemcpyDeviceToHost) stats[kD2h]++;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind kind, hipStream_t) {
    return hipMemcpy(d, s, n, kind);
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = a_handle<hipStream_t>(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    if (capturing) return stats[kMisuse]++, hipErrorStreamCaptureUnsupported;
    return stats[kSyncs]++, hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    capturing = false;
    return *g = a_handle<hipGraph_t>(), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *e = a_handle<hipGraphExec_t>(), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) { return *e = a_handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

hipError_t hipModuleLoad(hipModule_t* m, const char*) { return *m = a_handle<hipModule_t>(), hipSuccess; }
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
// Every kernel name is there.
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char*) {
    return *f = a_handle<hipFunction_t>(), hipSuccess;
}
hipError_t hipFuncGetAttribute(int* v, hipFunction_attribute a, hipFunction_t) {
    return *v = a == HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK ? 1024 : 0, hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 hipStream_t, void**, void**) {
    return hipSuccess;
}
}

hipError_t zlm_static_scratch_address(float** p) { return *p = nullptr, hipErrorInvalidSymbol; }
