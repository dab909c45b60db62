// A HIP runtime without a GPU, loaded (globally) before the library by
// tests/test_alloc_failure.py: device memory is host memory, launches run
// nothing and are recorded, and one allocation of a chosen size can be made to
// fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

static std::map<const void*, std::string> kernels;
static std::set<void*> live;
static size_t fail_size = 0;
static std::string watch;
static int watch_arg = 0;
static void* seen = nullptr;
static int launches = 0;

extern "C" {
// the next hipMalloc of exactly `bytes` fails
void fake_fail(size_t bytes) { fail_size = bytes; }
// record pointer argument `arg` of launches of kernels whose name contains `name`
void fake_watch(const char* name, int arg) {
    watch = name;
    watch_arg = arg;
    seen = nullptr;
    launches = 0;
}
int fake_launches() { return launches; }
// whether the recorded pointer is an allocation that still stands
int fake_seen_live() { return live.count(seen) != 0; }

hipError_t hipMalloc(void** p, size_t n) {
    *p = nullptr;
    if (fail_size && n == fail_size) {
        fail_size = 0;
        return hipErrorOutOfMemory;
    }
    *p = std::calloc(n ? n : 1, 1);
    live.insert(*p);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // R0600 in the header
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* symbol) {
    static std::map<const void*, void*> vars;
    if (!vars.count(symbol)) vars[symbol] = std::calloc(1, 1 << 24);
    *p = vars[symbol];
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void** args, size_t, hipStream_t) {
    if (!watch.empty() && kernels[f].find(watch) != std::string::npos) {
        ++launches;
        seen = *static_cast<void**>(args[watch_arg]);
    }
    return hipSuccess;
}
static dim3 cfg_grid, cfg_block;
static size_t cfg_shmem;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) {
    cfg_grid = g, cfg_block = b, cfg_shmem = s, cfg_stream = st;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
    *g = cfg_grid, *b = cfg_block, *s = cfg_shmem, *st = cfg_stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* module = nullptr;
    return &module;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned int, void*, void*, void*, void*,
                           int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}
}
