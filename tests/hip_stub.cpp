// A HIP runtime without a device, for tests of the library's host side on the CPU: allocations are
// address ranges (never touched, so of any size), copies and launches are only written down.
// Load it RTLD_GLOBAL before libprism_hip.so, whose HIP calls then resolve here.
#include <hip/hip_runtime.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Range {
    size_t bytes;
    hipMemoryType type;
};
std::map<uintptr_t, Range> g_ranges;
std::map<const void *, std::string> g_kernels;
std::vector<std::string> g_log;
std::string g_note;
bool g_capturing = false;
size_t g_largest = ~size_t(0);
uintptr_t g_handle = 0x1000;
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} g_config;

template <typename... A>
void note(const char *f, A... a) {
    char m[512];
    std::snprintf(m, sizeof m, f, a...);
    g_log.push_back(m);
}
const Range *find(const void *p) {
    auto it = g_ranges.upper_bound(reinterpret_cast<uintptr_t>(p));
    if (it == g_ranges.begin()) return nullptr;
    --it;
    return reinterpret_cast<uintptr_t>(p) < it->first + it->second.bytes ? &it->second : nullptr;
}
hipError_t reserve(void **p, size_t bytes, hipMemoryType type, const char *what) {
    if (bytes > g_largest) return hipErrorOutOfMemory;
    void *m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    g_ranges[reinterpret_cast<uintptr_t>(m)] = Range{bytes, type};
    note("%s %p %zu", what, m, bytes);
    *p = m;
    return hipSuccess;
}
hipError_t release(void *p, const char *what) {
    auto it = g_ranges.find(reinterpret_cast<uintptr_t>(p));
    if (it == g_ranges.end()) return hipErrorInvalidValue;
    note("%s %p", what, p);
    munmap(p, it->second.bytes);
    g_ranges.erase(it);
    return hipSuccess;
}
template <typename T>
hipError_t handle(T *h) {
    *h = reinterpret_cast<T>(g_handle += 16);
    return hipSuccess;
}
}  // namespace

extern "C" {

// The test's side.
void stub_capture(int on) { g_capturing = on != 0; }
void stub_largest(size_t bytes) { g_largest = bytes; }
int stub_alive(void *p) { return find(p) != nullptr; }
size_t stub_allocations() { return g_ranges.size(); }
const char *stub_log() {
    g_note.clear();
    for (const std::string &s : g_log) g_note += s + "\n";
    g_log.clear();
    return g_note.c_str();
}

// The runtime's.
void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(&g_handle); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t s) {
    g_config = {grid, block, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *s) {
    *grid = g_config.grid, *block = g_config.block, *shared = g_config.shared, *s = g_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **, size_t shared, hipStream_t s) {
    note("launch %s grid %u %u %u block %u lds %zu stream %p", g_kernels[f].c_str(), grid.x, grid.y, grid.z, block.x, shared,
         static_cast<void *>(s));
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return reserve(p, 64u << 20, hipMemoryTypeDevice, "symbol"); }
hipError_t hipMalloc(void **p, size_t bytes) { return reserve(p, bytes, hipMemoryTypeDevice, "malloc"); }
hipError_t hipFree(void *p) { return release(p, "free"); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return reserve(p, bytes, hipMemoryTypeHost, "host_malloc"); }
hipError_t hipHostFree(void *p) { return release(p, "host_free"); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::memset(a, 0, sizeof *a);
    const Range *r = find(p);
    if (!r) return hipErrorInvalidValue;
    a->type = r->type;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t s) {
    note("copy %p <- %p %zu stream %p", dst, src, bytes, static_cast<void *>(s));
    return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t bytes, hipMemcpyKind) {
    if (bytes <= 64) std::memcpy(dst, src, bytes);  // the error flag
    return hipSuccess;
}
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t *s) { return handle(s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *st) {
    *st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return g_capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return g_capturing = false, handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }

}  // extern "C"
