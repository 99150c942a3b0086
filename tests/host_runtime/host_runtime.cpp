// The part of the HIP runtime that the library calls, without a device: kernels are written down instead of run, memory is
// addresses out of a budget, streams are captured when a test says so.  Loaded in front of the library by tests/host_runtime.py.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdio>
#include <map>
#include <set>
#include <string>

namespace {
std::map<const void *, std::string> kernels;
std::set<void *> capturing;
std::string events;
size_t budget = (size_t)1 << 40, next_address = (size_t)1 << 44;
int cus = 256, masked_cus = 0;

void note(const char *format, ...) {
    char line[512];
    va_list args;
    va_start(args, format);
    vsnprintf(line, sizeof line, format, args);
    va_end(args);
    events += line;
    events += '\n';
}
}  // namespace

extern "C" {

const char *host_events() { return events.c_str(); }
void host_clear() { events.clear(); }
void host_budget(size_t bytes) { budget = bytes; }
void host_capture(void *stream, int on) {
    if (on) capturing.insert(stream);
    else capturing.erase(stream);
}
void host_masked_cus(int n) { masked_cus = n; }

void **__hipRegisterFatBinary(const void *) {
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) { kernels[host] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipErrorNotSupported; }

hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    *p = hipDeviceProp_t();
    p->multiProcessorCount = cus;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = (void *)((size_t)1 << 43), hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipErrorNotSupported; }
hipError_t hipDeviceSynchronize() { return note("synchronize"), hipSuccess; }

hipError_t hipMalloc(void **p, size_t bytes) {
    note("malloc %zu", bytes);
    if (bytes > budget) return hipErrorOutOfMemory;
    budget -= bytes;
    *p = (void *)next_address;
    next_address += (bytes + 255) / 256 * 256;
    return hipSuccess;
}
hipError_t hipFree(void *) { return hipSuccess; }

hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *status) {
    *status = capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipExtStreamGetCUMask(hipStream_t, uint32_t words, uint32_t *mask) {
    for (uint32_t i = 0; i < words; ++i) mask[i] = 0;
    const int n = masked_cus ? masked_cus : cus;
    for (int i = 0; i < n && i < (int)words * 32; ++i) mask[i / 32] |= 1u << (i % 32);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)&events, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { return note("record %p", (void *)s), hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) { return note("wait %p", (void *)s), hipSuccess; }

// (the first argument as an address: what the kernel that adds up a K split reads)
hipError_t hipLaunchKernel(const void *kernel, dim3 grid, dim3 block, void **args, size_t, hipStream_t s) {
    note("launch %s stream %p grid %u %u block %u first %p", kernels[kernel].c_str(), (void *)s, grid.x, grid.y, block.x, *(void **)args[0]);
    return hipSuccess;
}
}
