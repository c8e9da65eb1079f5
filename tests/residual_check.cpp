// Host check of the residual's first call (mr-lbm_amd/csrc/api.hip) when the
// pinned result buffer cannot be allocated: that call fails, and the next one
// is the first. The runtime calls on the way are replaced here, so no device
// is needed; kernels are not run. Prints "ok" and exits 0 on success.
#include <cstdio>
#include <cstdlib>

#include "../mr-lbm_amd/csrc/context.h"

static int pinned_calls = 0;

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (pinned_calls++ == 0) return hipErrorOutOfMemory;
    return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
}

int main() {
    mrlbm_ctx c{};
    c.N = 512;
    c.T = 512;
    c.ntiles = 1;
    c.initialised = true;
    double r = 0.0;
    const int failed = mrlbm_velocity_residual(&c, &r);
    const double held = c.device_bytes;
    const int first = mrlbm_velocity_residual(&c, &r);
    const double r1 = r;
    const int second = mrlbm_velocity_residual(&c, &r);
    if (failed != MRLBM_ENOMEM || held != 0.0 || first != MRLBM_OK || r1 != -1.0 || second != MRLBM_OK || r != 0.0) {
        std::printf("status %d %d %d, bytes %g, values %g %g\n", failed, first, second, held, r1, r);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
