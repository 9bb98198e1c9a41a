// A HIP runtime without a device, preloaded in front of the real one by test_launches.py: memory is host memory, kernels do
// not run, and every launch, copy and wait is written down.  It shows on the CPU which kernels a call takes and what it does
// when one of them fails.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string>& names()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::string g_log;
int g_fail_in = 0;             // the n-th launch from now fails
hipError_t g_error = hipSuccess;
dim3 g_grid, g_block;
size_t g_lds;
hipStream_t g_stream;

void note(const char* what, size_t bytes)
{
    g_log += std::string(what) + " " + std::to_string(bytes) + "\n";
}
}  // namespace

extern "C" {
const char* stub_log() { return g_log.c_str(); }
void stub_clear() { g_log.clear(); }
void stub_fail_launch(int n) { g_fail_in = n; }

void** __hipRegisterFatBinary(const void*)
{
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned int, void*, void*, dim3*, dim3*, int*) { names()[host] = name; }
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    g_grid = grid, g_block = block, g_lds = lds, g_stream = stream;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = g_grid, *block = g_block, *lds = g_lds, *stream = g_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3 block, void**, size_t lds, hipStream_t)
{
    char dims[96];
    std::snprintf(dims, sizeof(dims), " %u %u %u %u %zu", grid.x, grid.y, grid.z, block.x, lds);
    const bool fails = g_fail_in > 0 && --g_fail_in == 0;
    if (fails) g_error = hipErrorLaunchFailure;
    g_log += (fails ? "failed " : "launch ") + names()[host] + dims + "\n";
    return fails ? g_error : hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_error;
    g_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* dev) { return *dev = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)       // (the header names the versioned symbol)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 64 * 1024;
    p->sharedMemPerBlockOptin = 160 * 1024;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n)
{
    note("malloc", n);
    return *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096), hipSuccess;
}
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int)
{
    note("pinned", n);
    return *p = std::aligned_alloc(4096, (n + 4095) / 4096 * 4096), hipSuccess;
}
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    note("copy", n);
    return std::memcpy(d, s, n), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return note("wait", 0), hipSuccess; }
}
