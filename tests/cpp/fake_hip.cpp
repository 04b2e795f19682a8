// fake_hip.cpp -- a host stand-in for the HIP runtime calls that the library's
// key loading and context code make, for tests of their failure paths on a
// machine without a GPU: device memory is malloc'd, copies and kernels do
// nothing, and one call by name can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <set>

namespace {
char g_name[64];
int g_after = -1;  // calls of g_name that still succeed; -1: none fails
std::set<void *> g_live;

hipError_t call(const char *name)
{
    if (g_after < 0 || std::strcmp(name, g_name) != 0) return hipSuccess;
    if (g_after-- > 0) return hipSuccess;
    return std::strcmp(name, "hipMalloc") ? hipErrorUnknown : hipErrorOutOfMemory;
}

hipError_t take(const char *name, void **p, size_t n)
{
    *p = nullptr;
    if (hipError_t e = call(name)) return e;
    *p = std::malloc(n);
    g_live.insert(*p);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}

hipError_t give(void *p)
{
    if (!p) return hipSuccess;
    if (!g_live.erase(p)) std::abort();  // not allocated, or given back twice
    std::free(p);
    return hipSuccess;
}

char g_handle;
template <class H>
hipError_t handle(const char *name, H *h)
{
    *h = reinterpret_cast<H>(&g_handle);
    return call(name);
}
}  // namespace

extern "C" {

// the call of `name` after `after` more successful ones fails (once)
void fake_fail(const char *name, int after)
{
    std::strncpy(g_name, name, sizeof g_name - 1);
    g_after = after;
}
int fake_pending() { return g_after >= 0; }
int fake_live() { return int(g_live.size()); }

hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return take("hipMalloc", p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return take("hipHostMalloc", p, n); }
hipError_t hipFree(void *p) { return give(p); }
hipError_t hipHostFree(void *p) { return give(p); }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return call("hipMemcpy"); }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t)
{
    return call("hipMemcpyAsync");
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t)
{
    return call("hipLaunchKernel");
}
hipError_t hipGetLastError() { return call("hipGetLastError"); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle("hipStreamCreateWithFlags", s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return call("hipStreamSynchronize"); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return call("hipStreamBeginCapture"); }
hipError_t hipEventCreate(hipEvent_t *e) { return handle("hipEventCreate", e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle("hipEventCreateWithFlags", e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return call("hipEventRecord"); }
hipError_t hipEventSynchronize(hipEvent_t) { return call("hipEventSynchronize"); }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    *p = &g_handle;
    return hipSuccess;
}

}  // extern "C"
