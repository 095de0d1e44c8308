// A HIP runtime without a device, for tests of the library's host code: device memory is
// zeroed host memory, copies are memcpy, kernels are not run. Loaded with global symbols
// before libpbrtm.so it takes the place of the HIP runtime there. Every kernel launch and
// graph launch is reported to a hook, which may write into "device" memory (kernel
// arguments are passed on as the array of pointers that hipLaunchKernel gets) and whose
// non-zero result is returned as the call's error.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {

using LaunchHook = int (*)(const char *kernel, uint32_t blocks, uint32_t threads, int captured, void **args);
using GraphHook = int (*)();
using OccupancyHook = int (*)(const char *kernel);

LaunchHook g_launch = nullptr;
GraphHook g_graph = nullptr;
OccupancyHook g_occupancy = nullptr;
size_t g_fail_copy = 0;  // the next copy of this many bytes fails
bool g_capturing = false;
hipError_t g_last = hipSuccess;

std::map<const void *, std::string> &kernels() {
    static std::map<const void *, std::string> m;
    return m;
}
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_config;

template <typename T> T handle() {
    return reinterpret_cast<T>(std::calloc(1, 64));
}

hipError_t note(int code) {
    if (code != 0) g_last = hipError_t(code);
    return hipError_t(code);
}

}  // namespace

extern "C" {

void fake_hip_hooks(LaunchHook launch, GraphHook graph, OccupancyHook occupancy) {
    g_launch = launch;
    g_graph = graph;
    g_occupancy = occupancy;
}
void fake_hip_fail_copy(uint64_t bytes) { g_fail_copy = bytes; }

void **__hipRegisterFatBinary(const void *) { return handle<void **>(); }
void __hipUnregisterFatBinary(void **p) { std::free(p); }
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    kernels()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream) {
    g_config = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream) {
    *grid = g_config.grid;
    *block = g_config.block;
    *lds = g_config.lds;
    *stream = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t) {
    return note(g_launch ? g_launch(kernels()[f].c_str(), grid.x, block.x, g_capturing, args) : 0);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return note(g_graph ? g_graph() : 0); }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int, size_t) {
    *n = g_occupancy ? g_occupancy(kernels()[f].c_str()) : 1;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "fake HIP error"; }

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *mem = std::calloc(1, 64 << 20);
    return *p = mem, hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t) {
    if (g_fail_copy != 0 && n == g_fail_copy) {
        g_fail_copy = 0;
        return hipErrorUnknown;
    }
    return std::memcpy(dst, src, n), hipSuccess;
}
hipError_t hipMemsetAsync(void *dst, int v, size_t n, hipStream_t) { return std::memset(dst, v, n), hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = handle<hipStream_t>(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(reinterpret_cast<void *>(s)), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return g_capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) {
    g_capturing = false;
    return *g = handle<hipGraph_t>(), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    return *x = handle<hipGraphExec_t>(), hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free(reinterpret_cast<void *>(g)), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return std::free(reinterpret_cast<void *>(x)), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(reinterpret_cast<void *>(e)), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.f, hipSuccess; }

}  // extern "C"
