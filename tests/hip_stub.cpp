// Stand-in for the HIP runtime, preloaded under libfdtd_hip.so on a machine
// without a GPU, for tests of the host code alone: which kernels a call
// launches, in which shape, and what it does when a launch fails.  Device
// memory is host memory, kernels do not run, and every launch appends
//   kernel name (demangled, no arguments) <tab> grid x y z <tab> block x y z
// to the file HIP_STUB_LOG.  After stub_fail_launch(n) the n-th launch from
// then on returns an error once; after stub_queue(ms) the next synchronisation
// of a stream takes so long.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <utility>

#include "../fdtd-cuda_amd/csrc/sim.h"

namespace {
// made on first use: kernels are registered before this library's own static objects are set up
std::map<const void *, std::string> &names() {
    static auto *m = new std::map<const void *, std::string>;
    return *m;
}
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_stream;
hipError_t g_last = hipSuccess;
long g_fail = -1;
int g_queued_ms = 0, g_waits = 0;
char g_handle[8];
template <typename T>
hipError_t handle(T *out) {
    *out = (T)(void *)g_handle;
    return hipSuccess;
}
template <typename T>
hipError_t alloc(T *out, size_t n) {
    *out = (T)std::calloc(n ? n : 1, 1);   // large blocks are untouched zero pages
    return *out ? hipSuccess : hipErrorOutOfMemory;
}
}  // namespace

extern "C" {

void stub_fail_launch(long n) { g_fail = n; }
void stub_queue(int ms) { g_queued_ms = ms; }
int stub_waits(void) { return g_waits; }   // stream synchronisations so far
// Records of a point monitor or objective probe that the handle still holds for a later launch.
int stub_pending_records(const fdtd_sim *s) { return (s->rec_dst[0] != nullptr) + (s->rec_dst[1] != nullptr); }

void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    int st = 0;
    char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    std::string n = d ? d : name;
    std::free(d);
    for (const char *p : {"void ", "(anonymous namespace)::"})
        if (n.rfind(p, 0) == 0) n = n.substr(std::strlen(p));
    names()[host] = n.substr(0, n.find('('));
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
    g_grid = g; g_block = b; g_shmem = sh; g_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
    *g = g_grid; *b = g_block; *sh = g_shmem; *st = g_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t) {
    if (g_fail > 0 && --g_fail == 0) return g_last = hipErrorLaunchFailure;
    static FILE *log = std::getenv("HIP_STUB_LOG") ? std::fopen(std::getenv("HIP_STUB_LOG"), "a") : nullptr;
    if (log) {
        std::fprintf(log, "%s\t%u %u %u\t%u %u %u\n", names()[f].c_str(), g.x, g.y, g.z, b.x, b.y, b.z);
        std::fflush(log);
    }
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return alloc(p, n); }
hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = nullptr; return hipErrorInvalidSymbol; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }   // no kernel runs: memory is as allocated
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    g_waits++;
    std::this_thread::sleep_for(std::chrono::milliseconds(std::exchange(g_queued_ms, 0)));
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }

}  // extern "C"
