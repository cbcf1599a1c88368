#include "fake_hip.hpp"

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>

namespace fake {
std::function<void(const Launch &)> on_launch;
std::string refuse;
bool refuse_attributes = false;
size_t memory = size_t(1) << 33, used = 0, peak = 0;
}  // namespace fake

namespace {

std::map<const void *, std::string> &kernels() {
    static std::map<const void *, std::string> names;
    return names;
}
std::map<void *, size_t> &blocks() {
    static std::map<void *, size_t> sizes;
    return sizes;
}
hipError_t last = hipSuccess;

// As the runtime does: a failure stays until hipGetLastError reports it.
hipError_t result(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}

struct Config {
    dim3 grid, block;
    size_t shared = 0;
    hipStream_t stream = nullptr;
} config;

hipError_t launch(const void *f, dim3 grid, dim3 block, void **args) {
    const std::string &name = kernels()[f];
    if (!fake::refuse.empty() && name.find(fake::refuse) != std::string::npos)
        return result(hipErrorInvalidConfiguration);
    if (grid.x == 0 || grid.y == 0 || block.x == 0) return result(hipErrorInvalidConfiguration);
    if (fake::on_launch) fake::on_launch(fake::Launch{name, grid, block, args});
    return hipSuccess;
}

}  // namespace

size_t fake::size_of(const void *p) { return blocks()[const_cast<void *>(p)]; }

namespace {

template <class T>
hipError_t handle(T *out) {
    *out = reinterpret_cast<T>(std::malloc(1));
    return hipSuccess;
}

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    kernels()[f] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
    config = {grid, block, shared, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = config.grid;
    *block = config.block;
    *shared = config.shared;
    *stream = config.stream;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t) {
    return launch(f, grid, block, args);
}
hipError_t hipExtLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t, hipStream_t, hipEvent_t,
                              hipEvent_t, int) {
    return launch(f, grid, block, args);
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) {
    return result(fake::refuse_attributes ? hipErrorInvalidValue : hipSuccess);
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 4;
    return hipSuccess;
}
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "refused by the test"; }

hipError_t hipMalloc(void **p, size_t n) {
    if (fake::used + n > fake::memory) return result(hipErrorOutOfMemory);
    *p = std::calloc(n, 1);
    blocks()[*p] = n;
    fake::used += n;
    fake::peak = std::max(fake::peak, fake::used);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    fake::used -= blocks()[p];
    blocks().erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) {
    std::memmove(to, from, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) {
    std::memmove(to, from, n);
    return hipSuccess;
}
hipError_t hipMemset(void *p, int v, size_t n) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) {
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t p, int v, size_t n, hipStream_t) {
    for (size_t i = 0; i < n; ++i) static_cast<int *>(p)[i] = v;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static int scratch[65536];
    *p = scratch;
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 163840;
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t s) {
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) {
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    std::free(e);
    return hipSuccess;
}

}  // extern "C"
