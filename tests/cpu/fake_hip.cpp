// A model of the HIP runtime calls that the launcher (maize_amd/csrc/shim.cpp) makes, for tests without a device: memory is a
// counter of addresses, a launch is a line in a log.  It keeps to the rules that matter to a launcher under stream capture:
//   * waiting for a captured stream is an error and spoils the capture;
//   * hipMalloc and hipFree while a stream is captured are errors that spoil the capture, unless the calling thread's capture
//     mode is relaxed;
//   * what is launched or set on a captured stream becomes a node: a kernel node holds the address of its workspace.
// Log lines: "malloc <address> <bytes>", "free <address>", "wait <stream>", "set <stream> <address> <bytes>" and
// "launch <stream> <kernel> <grid> <ksplit> <workspace>", with "node " in front where it was recorded.
#include <hip/hip_runtime.h>

#include <cinttypes>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>

#include "maize_hip.h"
#include "noalloc.hpp"

namespace {
std::string g_log;
uint64_t g_next = 1ull << 32;
size_t g_limit = ~(size_t)0, g_used = 0;                     // device memory
std::map<uint64_t, size_t> g_live;
std::map<void*, hipStreamCaptureStatus> g_captured;          // streams being captured
hipStreamCaptureMode g_mode = hipStreamCaptureModeGlobal;    // the thread's
hipError_t g_last = hipSuccess;

hipError_t ret(hipError_t e) { if (e != hipSuccess) g_last = e; return e; }
template <class... T> void say(const char* fmt, T... x) {
    char b[256];
    snprintf(b, sizeof b, fmt, x...);
    g_log += b;
}
bool is_captured(hipStream_t s) { return g_captured.count(s) != 0; }
bool unsafe_call() {                                         // one that a capture does not allow
    if (g_captured.empty() || g_mode == hipStreamCaptureModeRelaxed) return false;
    for (auto& kv : g_captured) kv.second = hipStreamCaptureStatusInvalidated;
    return true;
}
}  // namespace

extern "C" {
extern const unsigned char maize_embedded_hsaco[1] = {0};
extern const unsigned char maize_embedded_hsaco_end[1] = {0};
extern const unsigned char maize_embedded_forms[1] = {0};

// ---- the test's side ----
const char* fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
void fake_memory(size_t bytes) { g_limit = bytes; }
void fake_capture(void* s) { g_captured[s] = hipStreamCaptureStatusActive; }
int fake_end_capture(void* s) {                              // 1: the capture is whole
    const int ok = g_captured[s] == hipStreamCaptureStatusActive;
    g_captured.erase(s);
    return ok;
}
int fake_relaxed() { return g_mode == hipStreamCaptureModeRelaxed; }

// ---- the launcher's side ----
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 163840;
    p->warpSize = 64;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error of the model"; }
hipError_t hipGetLastError() { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) {
    if (unsafe_call()) return ret(hipErrorStreamCaptureUnsupported);
    if (g_used + n > g_limit) return ret(hipErrorOutOfMemory);
    *p = (void*)g_next;
    g_live[g_next] = n;
    say("malloc %" PRIu64 " %zu\n", g_next, n);
    g_used += n;
    g_next += (n + 0xFFFFu) & ~0xFFFFull;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (unsafe_call()) return ret(hipErrorStreamCaptureUnsupported);
    auto it = g_live.find((uint64_t)p);
    if (it == g_live.end()) return ret(hipErrorInvalidValue);
    g_used -= it->second;
    g_live.erase(it);
    say("free %" PRIu64 "\n", (uint64_t)p);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* p, int, size_t n, hipStream_t s) {
    say("%sset %" PRIu64 " %" PRIu64 " %zu\n", is_captured(s) ? "node " : "", (uint64_t)s, (uint64_t)p, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    if (is_captured(s)) {
        g_captured[s] = hipStreamCaptureStatusInvalidated;
        return ret(hipErrorStreamCaptureUnsupported);
    }
    say("wait %" PRIu64 "\n", (uint64_t)s);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    if (!s && !g_captured.empty()) return ret(hipErrorStreamCaptureImplicit);
    *st = is_captured(s) ? g_captured[s] : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) { std::swap(*m, g_mode); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)g_next; g_next += 0x10000; return hipSuccess; }
hipError_t hipStreamCreate(hipStream_t* s) { return hipStreamCreateWithFlags(s, 0); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipModuleLoadData(hipModule_t* m, const void*) { *m = (hipModule_t)1; return hipSuccess; }
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) { *f = (hipFunction_t)strdup(name); return hipSuccess; }
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by, unsigned bz, unsigned, hipStream_t s,
                                 void**, void** extra) {
    // a launch's work items are counted in 32 bits
    if ((uint64_t)gx * bx >> 32 || (uint64_t)gy * by >> 32 || (uint64_t)gz * bz >> 32) return ret(hipErrorInvalidConfiguration);
    if (is_captured(s) && g_captured[s] != hipStreamCaptureStatusActive) return ret(hipErrorStreamCaptureInvalidated);
    maize_gemm_args_t a;
    memset(&a, 0, sizeof a);
    if (*(size_t*)extra[3] == sizeof a) memcpy(&a, extra[1], sizeof a);
    say("%slaunch %" PRIu64 " %s %" PRIu64 " %u %" PRIu64 "\n", is_captured(s) ? "node " : "", (uint64_t)s, (const char*)f, (uint64_t)gx * gy * gz, a.ksplit,
        (uint64_t)a.workspace);
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
}  // extern "C"

namespace maize {
hipError_t noalloc_scratch(int, void** p, size_t* n) {
    *p = (void*)(1ull << 24);
    *n = MAIZE_NOALLOC_SCRATCH_BYTES;
    return hipSuccess;
}
}  // namespace maize
