// hipMalloc that reports no memory for one chosen request and its repeat
// without headroom, and is the runtime's own otherwise.  Loaded with
// RTLD_GLOBAL before libpagani.
#include <dlfcn.h>

#include <cstddef>

static int requests = 0, fail_at = 0;
static size_t failed = 0;

extern "C" {
void malloc_fails(int nth) { requests = 0, fail_at = nth, failed = 0; }  // 1: the next request; 0: none
int malloc_requests() { return requests; }

int hipMalloc(void **p, size_t bytes)
{
    static auto real = (int (*)(void **, size_t))dlsym(dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL), "hipMalloc");
    if (failed != 0 && bytes < failed) return failed = 0, 2;  // hipErrorOutOfMemory
    if (++requests == fail_at) return failed = bytes, 2;
    failed = 0;
    return real(p, bytes);
}
}
