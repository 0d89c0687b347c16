// hip_stub.cpp — the HIP runtime entry points that the library uses, for a CPU build in
// which nothing runs: a kernel launch is recorded (kernel, grid, block) and device memory
// is an address that nobody may read.  Launches whose grid is past the runtime's limit of
// 2^32 work-items per dimension are refused as the runtime refuses them.  The library's
// own objects are linked against this, so what is recorded is its dispatch.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
std::mutex mu;
std::map<const void*, std::string>& names() {
    static auto* m = new std::map<const void*, std::string>;
    return *m;
}
std::string log_;
hipError_t last = hipSuccess;
size_t malloc_limit = ~size_t(0);
bool capturing = false;
int pointer_device = -1;                // of memory that the library does not own; -1: not known
uintptr_t next_address = uintptr_t(1) << 44;

struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
thread_local std::vector<Config> configs;
}  // namespace

extern "C" {
// ---- what the tests set and read
void stub_malloc_limit(size_t bytes) { malloc_limit = bytes; }
void stub_capturing(int on) { capturing = on != 0; }
void stub_pointer_device(int d) { pointer_device = d; }
// The launches since the last call, one per line: kernel|grid x y z|block.  Freed by the caller.
char* stub_launches() {
    std::lock_guard<std::mutex> g(mu);
    char* s = strdup(log_.c_str());
    log_.clear();
    return s;
}

// ---- registration and launches
void** __hipRegisterFatBinary(const void*) { return (void**)calloc(1, sizeof(void*)); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
    int status = 0;
    char* n = abi::__cxa_demangle(device, nullptr, nullptr, &status);
    names()[host] = n ? n : device;
    free(n);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, hipStream_t s) {
    configs.push_back({g, b, shmem, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shmem, hipStream_t* s) {
    const Config c = configs.back();
    configs.pop_back();
    *g = c.grid; *b = c.block; *shmem = c.shmem; *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t) {
    const uint64_t lim = uint64_t(1) << 32;
    if (!g.x || !g.y || !g.z || uint64_t(g.x) * b.x >= lim || uint64_t(g.y) * b.y >= lim || uint64_t(g.z) * b.z >= lim ||
        uint64_t(b.x) * b.y * b.z > 1024)
        return last = hipErrorInvalidConfiguration;
    char tail[128];
    snprintf(tail, sizeof tail, "|%u %u %u|%u\n", g.x, g.y, g.z, b.x * b.y * b.z);
    std::lock_guard<std::mutex> l(mu);
    log_ += names()[f] + tail;
    return hipSuccess;
}

// ---- device, memory, streams
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }   // the CUs
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes > malloc_limit) return last = hipErrorOutOfMemory;
    std::lock_guard<std::mutex> g(mu);
    *p = (void*)next_address;
    next_address += (bytes + 4095) / 4096 * 4096;
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = calloc(1, bytes);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return hipMalloc(p, 4096); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*) {
    if (pointer_device < 0) return last = hipErrorInvalidValue;
    a->type = hipMemoryTypeDevice;
    a->device = pointer_device;
    return hipSuccess;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}
