// A HIP runtime on the CPU for host-path tests: device memory is host memory within a budget, copies
// are memcpy, kernels do nothing.  Linked into a test program it takes the place of the runtime's
// functions that libmdgfx950.so calls.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

size_t g_budget = ~(size_t)0, g_used = 0;  // bytes of device memory
int g_refused = 0;                         // allocations that did not fit
static hipError_t g_last = hipSuccess;
static std::map<void*, size_t> g_sizes;
static std::mutex g_lock;

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    std::lock_guard<std::mutex> hold(g_lock);
    if (n > g_budget - g_used) {
        g_refused++;
        *p = nullptr;
        return g_last = hipErrorOutOfMemory;
    }
    *p          = calloc(n ? n : 1, 1);
    g_sizes[*p] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    std::lock_guard<std::mutex> hold(g_lock);
    auto it = g_sizes.find(p);
    if (it == g_sizes.end()) return p ? g_last = hipErrorInvalidValue : hipSuccess;
    g_used -= it->second;
    g_sizes.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = calloc(n, 1);
    return hipSuccess;
}
hipError_t hipHostFree(void* p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* m, hipStream_t* s)
{
    *g = *b = dim3(1);
    *m = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last             = hipSuccess;
    return e;
}
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 256;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    *s = (hipStream_t)8;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = (hipEvent_t)8;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)8;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}
}
