/* hipHostMalloc that fails on request, for tests of what the library does without pinned memory: loaded
 * with RTLD_GLOBAL before libmdarap.so, it stands in front of the runtime's. A refused call also asks for a
 * device that does not exist, so the runtime keeps an error as its last one, as it does when it refuses. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

size_t shim_lo = 1, shim_hi = 0; /* sizes in [shim_lo, shim_hi] fail */
int shim_refused = 0;

int hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    void *hip = dlopen("libamdhip64.so.7", RTLD_LAZY);
    if (bytes < shim_lo || bytes > shim_hi)
        return ((int (*)(void **, size_t, unsigned))dlsym(hip, "hipHostMalloc"))(p, bytes, flags);
    ++shim_refused;
    *p = 0;
    ((int (*)(int))dlsym(hip, "hipSetDevice"))(1 << 20);
    return 2; /* hipErrorOutOfMemory */
}
