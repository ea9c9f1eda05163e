// A HIP runtime on host memory for tests of libpagani's host code without a
// GPU: two devices, allocations filled with 0xA5, copies and clears carried
// out, kernels not run but reported (name, current device, stream's device,
// arguments).  Loaded with RTLD_GLOBAL before libpagani, its symbols win over
// the runtime's.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Range {
    size_t bytes;
    int device;
    bool managed;
};
struct Stream {
    int device;
};
std::map<char *, Range> ranges;
std::map<const void *, std::string> kernels;
int current = 0, mallocs = 0, fail_at = 0, copies = 0;
void (*hook)(const char *, int, int, void **) = nullptr;
struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} config;
}  // namespace

extern "C" {
// the test's side
void stub_hook(void (*f)(const char *, int, int, void **)) { hook = f; }
void stub_fail_malloc(int nth) { mallocs = 0, fail_at = nth; }  // 1: the next one; 0: none
int stub_mallocs() { return mallocs; }
int stub_live() { return (int)ranges.size(); }
int stub_copies() { return copies; }
int stub_device() { return current; }
void *stub_alloc(size_t bytes, int device, int managed)
{
    char *p = (char *)std::malloc(bytes);
    std::memset(p, 0xA5, bytes);
    ranges[p] = Range{bytes, device, managed != 0};
    return p;
}

// the runtime's
hipError_t hipGetDeviceCount(int *n) { return *n = 2, hipSuccess; }
hipError_t hipSetDevice(int d) { return current = d, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 160 * 1024;
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t) new Stream{current}, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete (Stream *)s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = std::calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    // pg_buf asks again without headroom: a failing request fails both times
    static size_t again = 0;
    const bool repeat = again != 0 && n < again;
    if (!repeat && ++mallocs == fail_at) {
        again = n;
        return hipErrorOutOfMemory;
    }
    if (repeat) return again = 0, hipErrorOutOfMemory;
    *p = stub_alloc(n, current, 0);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    ranges.erase((char *)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    copies++;
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    for (auto &r : ranges)
        if ((char *)p >= r.first && (char *)p < r.first + r.second.bytes) {
            std::memset(a, 0, sizeof *a);
            a->type = r.second.managed ? hipMemoryTypeManaged : hipMemoryTypeDevice;
            a->device = r.second.device;
            a->isManaged = r.second.managed;
            return hipSuccess;
        }
    return hipErrorInvalidValue;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char room[8 << 20];
    return *p = room, hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 160 * 1024, hipSuccess; }

hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s)
{
    if (hook) hook(kernels[f].c_str(), current, s ? ((Stream *)s)->device : current, args);
    return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t m, hipStream_t s, hipEvent_t, hipEvent_t, int)
{
    return hipLaunchKernel(f, g, b, args, m, s);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, hipStream_t s) { return config = Config{g, b, m, s}, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, hipStream_t *s)
{
    *g = config.grid, *b = config.block, *m = config.shared, *s = config.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
