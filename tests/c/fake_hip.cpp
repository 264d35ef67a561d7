/*
 * A stand-in for the HIP runtime, for tests of the library's host side on a
 * machine without a GPU: device memory is host memory, kernels are recorded
 * instead of run.  Loaded with RTLD_GLOBAL before libchiml_amd.so, whose
 * calls then end here.
 *
 * What a test reads and sets: fake_hip_log() (one line per call of interest),
 * fake_hip_clear(), fake_hip_fail_size(bytes): hipMalloc of exactly that many
 * bytes fails from its second call on; fake_hip_refuse(n): the first n - 1
 * calls of hipMalloc from here on succeed, the others fail (0: none fails).
 * fake_hip_held(): bytes allocated and not freed.
 */
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::string g_log;
// (the library's kernels may be registered before this file's own start-up)
std::map<const void*, std::string>& names() {
    static auto* m = new std::map<const void*, std::string>;
    return *m;
}
size_t g_fail_size = 0;
int g_fail_seen = 0, g_refuse = 0;
size_t g_held = 0;
std::map<void*, size_t>& blocks() {
    static auto* m = new std::map<void*, size_t>;
    return *m;
}
bool g_capturing = false;
struct Call {
    dim3 g, b;
    size_t shm;
    hipStream_t s;
} g_call;
void put(const std::string& s) { g_log += s + "\n"; }
}  // namespace

extern "C" {
const char* fake_hip_log() { return g_log.c_str(); }
void fake_hip_clear() { g_log.clear(); }
void fake_hip_fail_size(size_t bytes) {
    g_fail_size = bytes;
    g_fail_seen = 0;
}
void fake_hip_refuse(int n) { g_refuse = n; }
size_t fake_hip_held() { return g_held; }

void** __hipRegisterFatBinary(const void*) {
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shm, hipStream_t s) {
    g_call = {g, b, shm, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shm, hipStream_t* s) {
    *g = g_call.g;
    *b = g_call.b;
    *shm = g_call.shm;
    *s = g_call.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void**, size_t shm, hipStream_t) {
    put((g_capturing ? "capture " : "launch ") + names()[fn] + " " + std::to_string(g.x) + " " + std::to_string(b.x) + " " + std::to_string(shm));
    return hipSuccess;
}
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
    std::memset(a, 0, sizeof *a);
    a->sharedSizeBytes = 16384;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* fn, hipFuncAttribute, int v) {
    put("attribute " + names()[fn] + " " + std::to_string(v));
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 160 * 1024;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (g_fail_size && n == g_fail_size && ++g_fail_seen > 1) {
        *p = nullptr;
        put("refused " + std::to_string(n));
        return hipErrorOutOfMemory;
    }
    if (g_refuse == 1) return hipErrorOutOfMemory;
    if (g_refuse > 1) --g_refuse;
    *p = std::calloc(n ? n : 1, 1);
    if (!*p) return hipErrorOutOfMemory;
    blocks()[*p] = n;
    g_held += n;
    return hipSuccess;
}
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return hipMalloc(p, n); }
hipError_t hipFree(void* p) {
    auto it = blocks().find(p);
    if (it != blocks().end()) {
        g_held -= it->second;
        blocks().erase(it);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipFreeAsync(void* p, hipStream_t) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char scratch[1 << 20];
    *p = scratch;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = nullptr;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    g_capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    g_capturing = false;
    *g = nullptr;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    static size_t n = 0;
    *e = reinterpret_cast<hipGraphExec_t>(++n);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
    put("graph " + std::to_string(reinterpret_cast<size_t>(e)));
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}
