// A stand-in for the HIP runtime calls that libvva.so makes, for CPU tests of
// its host code: kernel launches are recorded by name instead of run, memory
// is an address that nobody reads, and a test says whether the stream is
// under capture and how large an allocation still succeeds.  Loaded with
// RTLD_GLOBAL ahead of libvva.so, whose references then bind to it.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string>& kernels() {
    static std::map<const void*, std::string> m;
    return m;
}
std::string g_log;                       // one line per launch or allocation
bool g_capturing = false;
size_t g_malloc_max = (size_t)1 << 40;
uintptr_t g_next = (uintptr_t)1 << 44;   // 256-byte aligned addresses, never reused
hipError_t g_last = hipSuccess;
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_stream;
}  // namespace

extern "C" {

void fake_set(int capturing, size_t malloc_max) {
    g_capturing = capturing != 0;
    g_malloc_max = malloc_max;
}
// The log since the last call ("kernel <name>", "malloc <bytes>")
const char* fake_take_log() {
    static std::string out;
    out.swap(g_log);
    g_log.clear();
    return out.c_str();
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->name, "stand-in");
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (g_capturing) return g_last = hipErrorStreamCaptureUnsupported;
    if (n > g_malloc_max) return g_last = hipErrorOutOfMemory;
    g_log += "malloc " + std::to_string(n) + "\n";
    *p = (void*)g_next;
    g_next += (n + 255) / 256 * 256;
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = (void*)((uintptr_t)1 << 43); return hipSuccess; }
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void**, size_t, hipStream_t) {
    // "void vva::(anonymous namespace)::name<args>(...)" -> "name<args>"
    std::string n = kernels().count(f) ? kernels()[f] : "?";
    int st = 0;
    if (char* d = abi::__cxa_demangle(n.c_str(), nullptr, nullptr, &st)) {
        n = d;
        free(d);
    }
    const char* ns = "(anonymous namespace)::";
    if (const size_t at = n.find(ns); at != std::string::npos) n.erase(0, at + strlen(ns));
    n.erase(std::min(n.size(), n.find('(', n.find('>') == std::string::npos ? 0 : n.find('>'))));
    g_log += "kernel " + n + " grid " + std::to_string(grid.x) + "," + std::to_string(grid.y) + "," +
             std::to_string(grid.z) + "\n";
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
    g_grid = grid;
    g_block = block;
    g_shmem = shmem;
    g_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* s) {
    *grid = g_grid;
    *block = g_block;
    *shmem = g_shmem;
    *s = g_stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

}  // extern "C"
