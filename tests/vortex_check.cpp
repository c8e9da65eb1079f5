// Host check of the initial vortex (mr-lbm_amd/csrc/transfer.hip) when its
// kernel cannot be launched: the copy of its tables has ended before the
// tables are released. The runtime calls on the way are replaced here, so no
// device is needed; kernels are not run. Prints "ok" and exits 0 on success.
#include <cstdio>
#include <cstdlib>

#include "../mr-lbm_amd/csrc/context.h"

static bool copying = false, launched = false;

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFreeAsync(void* p, hipStream_t) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) {
    copying = true;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    copying = false;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) {
    launched = true;
    return hipErrorLaunchFailure;
}
hipError_t hipGetLastError(void) { return launched ? hipErrorLaunchFailure : hipSuccess; }
}

int main() {
    mrlbm_ctx c{};
    c.p.nx = c.p.ny = c.p.nz = 8;
    c.p.q = 19;
    c.p.rho0 = 1.0;
    c.bx = c.by = c.bz = 8;
    c.ntx = c.nty = c.ntz = c.ntiles = 1;
    c.T = 512;
    c.N = 512;
    const int rc = mrlbm_init_taylor_green(&c, 0.05, MRLBM_INIT_EQUILIBRIUM);
    if (rc != MRLBM_EHIP || !launched || copying) {
        std::printf("status %d, launched %d, copy under way %d\n", rc, launched, copying);
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
