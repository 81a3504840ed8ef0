/* A stand-in for the HIP runtime on the host: allocations are host memory,
 * launches do nothing, and every call that orders work is written to a log.
 * Loaded ahead of libesthera.so (RTLD_GLOBAL) it takes the place of the
 * runtime, so that the order in which the library enqueues its work, and what
 * it does when a call fails, can be tested without a GPU. */
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <unordered_map>

#include <hip/hip_runtime_api.h>

static std::string g_log, g_fail;
static hipError_t g_last = hipSuccess;
static std::unordered_map<const void*, std::string> g_kernels;
static uintptr_t g_handles = 0;
static dim3 g_grid, g_block;
static hipStream_t g_stream;
static size_t g_shmem;

/* a line of the log; the call fails if the line holds what fake_fail asked for */
static hipError_t say(const char* fmt, ...) {
    char line[512];
    va_list a;
    va_start(a, fmt);
    vsnprintf(line, sizeof(line), fmt, a);
    va_end(a);
    if (!g_fail.empty() && strstr(line, g_fail.c_str())) {
        g_fail.clear();
        g_log += std::string("failed ") + line + "\n";
        return g_last = hipErrorUnknown;
    }
    g_log += std::string(line) + "\n";
    return hipSuccess;
}
template <class H>
static int id(H h) { return (int)(uintptr_t)h; }

extern "C" {
const char* fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
void fake_fail(const char* what) { g_fail = what; }

void** __hipRegisterFatBinary(const void*) { return (void**)&g_handles; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
    g_grid = g, g_block = b, g_shmem = sh, g_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
    *g = g_grid, *b = g_block, *sh = g_shmem, *s = g_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t lds, hipStream_t s) {
    const std::string& name = g_kernels[f];
    if (name.find("6k_mtgp") != std::string::npos)   /* words and statuses of its steps: addresses and strides in bytes */
        return say("launch %s stream %d steps %d from %zu to %zu stride %llu words %zu stride %llu", name.c_str(), id(s),
                   *(int*)args[8], *(size_t*)args[2], *(size_t*)args[3], 4ull * *(uint64_t*)args[10], *(size_t*)args[6],
                   4ull * *(uint64_t*)args[9]);
    return say("launch %s stream %d grid %u lds %zu", name.c_str(), id(s), grid.x, lds);
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipFuncGetAttributes(hipFuncAttributes* a, const void*) {
    memset(a, 0, sizeof(*a));
    a->numRegs = 64;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { static char b[4096]; *p = b; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)288 << 30; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = malloc(n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = calloc(1, n);
    return say("hipHostMalloc %p bytes %zu", *p, n);
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return say("hipMemcpy"); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st) {
    memcpy(d, s, n);
    return say("hipMemcpyAsync stream %d", id(st));
}
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return say("hipMemset"); }
hipError_t hipDeviceSynchronize() { return say("hipDeviceSynchronize"); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)++g_handles; return say("stream %d", id(*s)); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return say("hipStreamSynchronize stream %d", id(s)); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return say("hipStreamWaitEvent stream %d event %d", id(s), id(e)); }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) { return say("hipStreamBeginCapture stream %d", id(s)); }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    *g = (hipGraph_t)++g_handles;
    return say("hipStreamEndCapture stream %d", id(s));
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    *x = (hipGraphExec_t)++g_handles;
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return say("hipGraphLaunch stream %d", id(s)); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) { *e = (hipEvent_t)++g_handles; return say("event %d flags %x", id(*e), f); }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return say("hipEventRecord event %d stream %d", id(e), id(s)); }
hipError_t hipEventSynchronize(hipEvent_t e) { return say("hipEventSynchronize event %d", id(e)); }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }
}
