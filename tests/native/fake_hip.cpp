// A HIP runtime on the CPU for host code under test: device memory is host memory that
// remembers its device, copies and fills run at once, kernels are not executed.  It
// counts what a second device would not survive: a launch, copy or fill on a
// stream while another device is current (kernels, fills) or with memory of another
// device.  Preloaded before libmdt_gpu.so.  FAKE_HIP_DEVICES: how many devices there are;
// FAKE_HIP_BYTES: memory of each (default unbounded); FAKE_HIP_BEST: which of the timings
// taken with events is the shortest.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
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
std::mutex mu;
std::map<uintptr_t, Block> blocks;
size_t used[8];
int current = 0;
int violations = 0, launches = 0;
std::string first;
struct Stream {
    int dev;
    bool capturing;
};

void violation(const char *what, int dev, int want) {
    if (!violations++) {
        char s[160];
        std::snprintf(s, sizeof s, "%s: device %d, the stream's is %d", what, dev, want);
        first = s;
    }
}
int device_of(const void *p) {
    std::lock_guard<std::mutex> l(mu);
    auto it = blocks.upper_bound((uintptr_t)p);
    if (it == blocks.begin()) return -1;
    --it;
    return (uintptr_t)p < it->first + it->second.bytes ? it->second.dev : -1;
}
void check(const char *what, const void *p, hipStream_t st) {
    const int d = device_of(p);
    if (d >= 0 && st && d != ((Stream *)st)->dev) violation(what, d, ((Stream *)st)->dev);
}
size_t limit() {
    const char *s = std::getenv("FAKE_HIP_BYTES");
    return s ? std::strtoull(s, nullptr, 10) : SIZE_MAX;
}
dim3 call_grid, call_block;
size_t call_shared;
hipStream_t call_stream;
}  // namespace

extern "C" {
int fake_hip_violations(char *what, int n) {
    if (what && n > 0) std::snprintf(what, n, "%s", first.c_str());
    return violations;
}
int fake_hip_launches() { return launches; }
long long fake_hip_used(int dev) { return (long long)used[dev]; }

void **__hipRegisterFatBinary(const void *) {
    static void *h;
    return &h;
}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    call_grid = g;
    call_block = b;
    call_shared = s;
    call_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *st) {
    *g = call_grid;
    *b = call_block;
    *s = call_shared;
    *st = call_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t st) {
    ++launches;
    if (st && ((Stream *)st)->dev != current) violation("kernel launch", current, ((Stream *)st)->dev);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    const char *s = std::getenv("FAKE_HIP_DEVICES");
    *n = s ? std::atoi(s) : 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    current = d;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    p->sharedMemPerBlock = 163840;
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes *a, const void *) {
    std::memset(a, 0, sizeof *a);
    a->sharedSizeBytes = 8192;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *s = std::calloc(1, 16 << 20);
    *p = s;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes) {
    if (bytes > limit() - used[current]) {
        *p = nullptr;
        return hipErrorOutOfMemory;
    }
    *p = std::calloc(1, bytes ? bytes : 1);
    std::lock_guard<std::mutex> l(mu);
    blocks[(uintptr_t)*p] = {bytes ? bytes : 1, current};
    used[current] += bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    {
        std::lock_guard<std::mutex> l(mu);
        auto it = blocks.find((uintptr_t)p);
        if (it != blocks.end()) {
            used[it->second.dev] -= it->second.bytes;
            blocks.erase(it);
        }
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    *p = std::calloc(1, bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) {
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
    check("copy", d, st);
    check("copy", s, st);
    std::memmove(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st) {
    check("fill", d, st);
    if (st && ((Stream *)st)->dev != current) violation("fill", current, ((Stream *)st)->dev);
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned) {
    *st = (hipStream_t) new Stream{current, false};
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t st) {
    delete (Stream *)st;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t st, hipStreamCaptureStatus *s) {
    *s = ((Stream *)st)->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode) {
    ((Stream *)st)->capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t *g) {
    ((Stream *)st)->capturing = false;
    *g = (hipGraph_t) new int(0);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    *e = (hipGraphExec_t) new int(0);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    delete (int *)g;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
    delete (int *)e;
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) {
    *e = (hipEvent_t) new int(current);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    delete (int *)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    static int n = 0;
    const char *best = std::getenv("FAKE_HIP_BEST");
    *ms = best && ++n == std::atoi(best) ? 0.5f : 1.0f;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake hip error"; }
hipError_t hipGetLastError() { return hipSuccess; }
}
