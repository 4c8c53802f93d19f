// A stand-in for the HIP runtime on the CPU, preloaded before the library under
// test: device memory is host memory, kernels do nothing, every call is written
// to a log, and a chosen call fails.  Host code of the library can thus be
// followed without a GPU.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

namespace {
std::recursive_mutex lock;
std::string log_text;
std::map<const void*, std::string> kernel_names;
std::map<void*, size_t> blocks;
std::string fail_call;      // the call that fails ...
int fail_in = 0;            // ... after so many more (1: the next), 0: none
hipError_t pending = hipSuccess;

void note(const std::string& s) {
    std::lock_guard<std::recursive_mutex> g(lock);
    log_text += s + "\n";
}
bool fails(const char* call) {
    std::lock_guard<std::recursive_mutex> g(lock);
    return fail_in > 0 && fail_call == call && --fail_in == 0;
}
std::string hex(const void* p) {
    char b[32];
    snprintf(b, sizeof(b), "%p", p);
    return b;
}
}  // namespace

extern "C" {
// ---- for the test
const char* standin_log() { return log_text.c_str(); }
void standin_clear() { log_text.clear(); }
void standin_fail(const char* call, int in) { fail_call = call; fail_in = in; }
// Bytes held, and their checksum.
size_t standin_bytes(uint64_t* sum) {
    size_t n = 0;
    *sum = 1469598103934665603ull;
    for (const auto& b : blocks) {
        n += b.second;
        for (size_t i = 0; i < b.second; ++i)
            *sum = (*sum ^ static_cast<unsigned char*>(b.first)[i]) * 1099511628211ull;
    }
    return n;
}

// ---- memory
hipError_t hipMalloc(void** p, size_t n) {
    if (fails("hipMalloc")) { note("hipMalloc failed"); *p = nullptr; return hipErrorOutOfMemory; }
    *p = calloc(1, n ? n : 1);
    blocks[*p] = n;
    note("hipMalloc");
    return hipSuccess;
}
hipError_t hipFree(void* p) { note("hipFree"); blocks.erase(p); free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }

// ---- device
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 163840 : 0;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { note("hipDeviceSynchronize"); return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = pending;
    pending = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }

// ---- events and captures
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = reinterpret_cast<hipEvent_t>(malloc(1)); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { note("record on " + hex(s)); return fails("hipEventRecord") ? hipErrorInvalidHandle : hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) { note("wait on " + hex(s)); return hipSuccess; }
static hipStream_t captured;
static unsigned long long capture_id;
void standin_capture(hipStream_t s, unsigned long long id) { captured = s; capture_id = id; }
hipError_t hipStreamGetCaptureInfo(hipStream_t s, hipStreamCaptureStatus* st, unsigned long long* id) {
    *st = captured && s == captured ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    *id = capture_id;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
    static hipStreamCaptureMode now = hipStreamCaptureModeGlobal;
    std::swap(*m, now);
    return hipSuccess;
}

// ---- kernels
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernel_names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { config = {g, b, lds, s}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = config.grid; *b = config.block; *lds = config.lds; *s = config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s) {
    if (fails("hipLaunchKernel") || (uint64_t)g.x * b.x >> 32 != 0) {   // (a launch takes fewer than 2^32 threads)
        note("failed launch");
        return pending = hipErrorLaunchFailure;
    }
    int bad = 0;
    char* plain = abi::__cxa_demangle(kernel_names[f].c_str(), nullptr, nullptr, &bad);
    std::string name = plain ? plain : kernel_names[f];
    free(plain);
    size_t end = std::min(name.find("_kernel") + 7, name.size()), at = end;
    while (at > 0 && (isalnum((unsigned char)name[at - 1]) || name[at - 1] == '_')) --at;
    note("launch " + name.substr(at, end - at) + " " + std::to_string(g.x) + " on " + hex(s));
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
}
