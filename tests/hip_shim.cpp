// Host-side stand-ins for a few HIP and thread calls, loaded (RTLD_GLOBAL)
// before libezlda.so, whose calls they then take: each passes its call on, or
// makes it fail, as the shim_* switches say.  Nothing reaches the device that
// would not have otherwise.
#include <dlfcn.h>

#include <cstdlib>
#include <system_error>
#include <thread>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

namespace {

template <class F>
F *real(const char *lib, const char *name) {
    void *h = dlopen(lib, RTLD_LAZY), *f = h ? dlsym(h, name) : nullptr;
    if (!f) std::abort();
    return reinterpret_cast<F *>(f);
}

#define HIP_CALL(name, ...) real<decltype(name)>("libamdhip64.so.7", #name)(__VA_ARGS__)

long launches_left = -1;   // launches until one fails; < 0: none does
size_t failing_bytes = 0;  // hipMalloc of exactly this much fails,
long failing_times = 0;    // this often
bool failing_pinned = false, failing_threads = false;
int cus = 0;
hipError_t pending = hipSuccess;

}  // namespace

extern "C" {

void shim_fail_launch(long after) { launches_left = after; }
long shim_launches_left() { return launches_left; }
void shim_fail_malloc(size_t bytes, long times) { failing_bytes = bytes, failing_times = times; }
void shim_fail_pinned(int on) { failing_pinned = on; }
void shim_fail_threads(int on) { failing_threads = on; }
void shim_cus(int n) { cus = n; }

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t st) {
    if (launches_left == 0) {
        launches_left = -1;
        return pending = hipErrorLaunchFailure;
    }
    if (launches_left > 0) --launches_left;
    return HIP_CALL(hipLaunchKernel, f, grid, block, args, lds, st);
}

hipError_t hipGetLastError() {
    const hipError_t e = HIP_CALL(hipGetLastError), p = pending;
    pending = hipSuccess;
    return p != hipSuccess ? p : e;
}

hipError_t hipMalloc(void **p, size_t bytes) {
    if (failing_times > 0 && bytes == failing_bytes) {
        --failing_times;
        return pending = hipErrorOutOfMemory;
    }
    return real<hipError_t(void **, size_t)>("libamdhip64.so.7", "hipMalloc")(p, bytes);
}

hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) {
    if (failing_pinned) return pending = hipErrorOutOfMemory;
    return real<hipError_t(void **, size_t, unsigned)>("libamdhip64.so.7", "hipHostMalloc")(p, bytes, flags);
}

hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int dev) {
    if (cus && a == hipDeviceAttributeMultiprocessorCount) {
        *v = cus;
        return hipSuccess;
    }
    return HIP_CALL(hipDeviceGetAttribute, v, a, dev);
}

}  // extern "C"

// what every std::thread starts with
void std::thread::_M_start_thread(_State_ptr state, void (*depend)()) {
    using Start = void(std::thread *, _State_ptr, void (*)());
    if (failing_threads) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    real<Start>("libstdc++.so.6", "_ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE")(
        this, std::move(state), depend);
}
