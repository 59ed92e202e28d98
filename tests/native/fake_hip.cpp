// The HIP calls libvta_hip's host code makes, on host memory and without a
// device: kernels are recorded and not run, copies are memcpy, streams are
// immediate.  Linked in place of libamdhip64 by the host-code tests.
#include "fake_hip.h"

#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <string>

namespace {
std::mutex g_mu;
std::condition_variable g_cv;
bool g_closed = false;
int g_waiting = 0;
size_t g_launches = 0, g_total = size_t(256) << 30;
std::set<std::string> g_names;   // node-based: their addresses stay
}  // namespace

void fake_hip_gate(bool closed) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_closed = closed;
    g_cv.notify_all();
}
void fake_hip_wait_for_waiter() {
    std::unique_lock<std::mutex> lk(g_mu);
    g_cv.wait(lk, [] { return g_waiting > 0; });
}
void fake_hip_memory(size_t bytes) { g_total = bytes; }
size_t fake_hip_launches() {
    std::lock_guard<std::mutex> lk(g_mu);
    return g_launches;
}

namespace vta {
void noalloc_setup(int) {}
}  // namespace vta

extern "C" {

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 64 << 10;
    p->maxSharedMemoryPerMultiProcessor = 160 << 10;
    p->maxThreadsPerBlock = 1024;
    p->maxGridSize[0] = 2147483647;
    p->maxGridSize[1] = p->maxGridSize[2] = 65536;
    for (int &d : p->maxThreadsDim) d = 1024;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = g_total; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
    *p = std::malloc(n ? n : 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    std::unique_lock<std::mutex> lk(g_mu);
    g_waiting += 1;
    g_cv.notify_all();
    g_cv.wait(lk, [] { return !g_closed; });
    g_waiting -= 1;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t *, size_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventCreate(hipEvent_t *) { return hipErrorNotSupported; }
hipError_t hipEventDestroy(hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipEventElapsedTime(float *, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }
hipError_t hipModuleLoad(hipModule_t *m, const char *) {
    *m = reinterpret_cast<hipModule_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipModuleUnload(hipModule_t m) { std::free(m); return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t, const char *name) {
    std::lock_guard<std::mutex> lk(g_mu);
    *f = reinterpret_cast<hipFunction_t>(const_cast<std::string *>(&*g_names.insert(name).first));
    return hipSuccess;
}
hipError_t hipFuncGetAttribute(int *v, hipFunction_attribute, hipFunction_t) {
    *v = 64;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 unsigned, unsigned, hipStream_t, void **, void **) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_launches += 1;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }

}  // extern "C"
