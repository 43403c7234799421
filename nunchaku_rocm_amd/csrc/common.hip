// Host-side pieces shared by every entry point: the per-thread error string and launch checking.
#include <stdarg.h>
#include <stdio.h>

#include <atomic>

#include "svdq_common.h"

namespace svdq {

static thread_local char g_err[512] = "";

void set_error(const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
}

int check_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("%s: HIP launch failed: %s", what, hipGetErrorString(e));
        return SVDQ_E_LAUNCH;
    }
    return SVDQ_OK;
}

int cu_count() {
    static std::atomic<int> cached{0};
    int n = cached.load(std::memory_order_relaxed);
    if (n > 0) return n;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
        n = 256;
    cached.store(n, std::memory_order_relaxed);
    return n;
}

}  // namespace svdq

extern "C" const char *svdq_last_error(void) { return svdq::g_err; }
extern "C" int svdq_abi_version(void) { return SVDQ_ABI_VERSION; }
