// Stand-in for the part of the HIP runtime that the library's host code calls,
// compiled by tests/test_host_runtime.py and loaded before the library: device
// memory is host memory, kernel launches do nothing, copies and fills are done at
// once but counted as pending on their stream until something waits for it.  As
// documented of HIP, hipMemset returns before the fill of device memory is done,
// and a non-blocking stream (every stream but the null one here) is not ordered
// with the null stream.
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<void*, int> pending;
std::map<std::string, int> calls;
size_t limit = ~(size_t)0;
struct Dim3 {
    unsigned x, y, z;
};
}  // namespace

extern "C" {

int host_pending(void* stream) { return pending[stream]; }
int host_calls(const char* name) { return calls[name]; }
// allocations above this many bytes fail
void host_malloc_limit(size_t bytes) { limit = bytes; }

int hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (n > limit) return 2;   // hipErrorOutOfMemory
    *p = malloc(n);
    memset(*p, 0xff, n);       // NaN
    return 0;
}
int hipFree(void* p)
{
    if (p != nullptr) ++calls["hipFree"];
    free(p);
    return 0;
}
int hipMemset(void* p, int v, size_t n)
{
    ++calls["hipMemset"];
    memset(p, v, n);
    ++pending[nullptr];
    return 0;
}
int hipMemsetAsync(void* p, int v, size_t n, void* s)
{
    ++calls["hipMemsetAsync"];
    memset(p, v, n);
    ++pending[s];
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int)
{
    memcpy(d, s, n);
    pending[nullptr] = 0;
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void* stream)
{
    ++calls["hipMemcpyAsync"];
    memcpy(d, s, n);
    ++pending[stream];
    return 0;
}
int hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, int, void* stream)
{
    ++calls["hipMemcpy2DAsync"];
    for (size_t r = 0; r < h; ++r) memcpy((char*)d + r * dp, (const char*)s + r * sp, w);
    ++pending[stream];
    return 0;
}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void*) { return 0; }
int __hipPopCallConfiguration(Dim3*, Dim3*, size_t*, void**) { return 0; }
int hipLaunchKernel(const void*, Dim3, Dim3, void**, size_t, void* stream)
{
    ++calls["hipLaunchKernel"];
    ++pending[stream];
    return 0;
}
int hipStreamSynchronize(void* s) { return pending[s] = 0; }
int hipDeviceSynchronize()
{
    pending.clear();
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { return *s = malloc(1), 0; }
int hipStreamDestroy(void* s) { return free(s), 0; }
int hipGetDevice(int* d) { return *d = 0; }
int hipDeviceGetAttribute(int* v, int, int) { return *v = 256, 0; }
int hipGetLastError() { return 0; }
const char* hipGetErrorString(int) { return "host stand-in error"; }

}  // extern "C"
