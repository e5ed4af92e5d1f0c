/* Host-side stand-ins for a few HIP and thread calls, loaded (RTLD_GLOBAL)
 * before libezlda.so, whose calls they then take: each passes its call on,
 * or makes it return an error, as the shim_* switches say.  Nothing reaches
 * the device that would not have otherwise. */
#define _GNU_SOURCE
#define __HIP_PLATFORM_AMD__ 1
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>
#include <stdlib.h>

#include <hip/hip_runtime_api.h>

static void *real(const char *name) {
    static void *lib;
    if (!lib) lib = dlopen("libamdhip64.so.7", RTLD_LAZY);
    void *f = lib ? dlsym(lib, name) : NULL;
    if (!f) abort();
    return f;
}

static long launches_left = -1;  /* launches until one fails; < 0: none does */
static size_t failing_bytes = 0; /* hipMalloc of exactly this much fails */
static int failing_pinned = 0, failing_threads = 0, cus = 0;
static hipError_t pending = hipSuccess;

void shim_fail_launch(long after) { launches_left = after; }
long shim_launches_left(void) { return launches_left; }
void shim_fail_malloc(size_t bytes) { failing_bytes = bytes; }
void shim_fail_pinned(int on) { failing_pinned = on; }
void shim_fail_threads(int on) { failing_threads = on; }
void shim_cus(int n) { cus = n; }

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t st) {
    if (launches_left == 0) {
        launches_left = -1;
        return pending = hipErrorLaunchFailure;
    }
    if (launches_left > 0) --launches_left;
    return ((hipError_t(*)(const void *, dim3, dim3, void **, size_t, hipStream_t))real("hipLaunchKernel"))(
        f, grid, block, args, lds, st);
}

hipError_t hipGetLastError(void) {
    const hipError_t e = ((hipError_t(*)(void))real("hipGetLastError"))(), p = pending;
    pending = hipSuccess;
    return p != hipSuccess ? p : e;
}

hipError_t hipMalloc(void **p, size_t bytes) {
    if (failing_bytes && bytes == failing_bytes) return pending = hipErrorOutOfMemory;
    return ((hipError_t(*)(void **, size_t))real("hipMalloc"))(p, bytes);
}

hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    if (failing_pinned) return pending = hipErrorOutOfMemory;
    return ((hipError_t(*)(void **, size_t, unsigned))real("hipHostMalloc"))(p, bytes, flags);
}

hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int dev) {
    if (cus && a == hipDeviceAttributeMultiprocessorCount) {
        *v = cus;
        return hipSuccess;
    }
    return ((hipError_t(*)(int *, hipDeviceAttribute_t, int))real("hipDeviceGetAttribute"))(v, a, dev);
}

int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    static int (*next)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    if (failing_threads) return EAGAIN;
    if (!next) next = (int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *))dlsym(RTLD_NEXT, "pthread_create");
    return next(t, a, f, arg);
}
