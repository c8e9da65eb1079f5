// Diagnostics on the device: node sampling (probe points and lines),
// per-moment FP64 means, a running mean flow and the turbulent kinetic
// energy against it. They replace the reference's treatData family
// (src/treatData.cu): mean_moment (:36-102), velocityProfile (:383-498) and
// probeExport (:501-584), which copy one node at a time to the host, the
// MEAN_FLOW accumulation of fMom_mean and turbulentKineticEnergy (:236-296).
// The field kernels take groups of four nodes and are bound by memory: FP32
// 192x160x128 moment sums 62.4 -> 28.0 us; FP16 512x256x256 mean flow (2.4 GB)
// 618 -> 463 us per call (5.2 TB/s), turbulent energy 435 -> 184 us. Taken row
// by row instead of patch by patch, the mean flow took 674 us.
#include <hip/hip_runtime.h>

#include <cstring>

#include "context.h"
#include "linear.h"
#include "transfer.h"

using namespace mrlbm;

namespace {

// stored-convention moments of n nodes (xyz triples) as FP64
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_sample(const void* mom_, Linear L, const int* __restrict__ xyz, int n,
                                                        double* __restrict__ out) {
    using W = Word<S>;
    const auto mom = gptr((const typename W::T*)mom_);
    const int k = blockIdx.x * RED_THREADS + threadIdx.x;
    if (k >= n) return;
    const size_t e = L.at((uint32_t)xyz[3 * (size_t)k], (uint32_t)xyz[3 * (size_t)k + 1], (uint32_t)xyz[3 * (size_t)k + 2]);
#pragma unroll
    for (int m = 0; m < 10; m++) out[10 * (size_t)k + m] = (double)W::dec(mom[e + (size_t)m * L.T], L.rscale[m]);
}

// per-workgroup FP64 sums of the 10 stored moments
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_moment_sums(const void* mom, BlockGroups g, Linear L,
                                                             double* __restrict__ partial) {
    double v[10] = {};
    for (uint32_t i = blockIdx.x * RED_THREADS + threadIdx.x; i < g.n; i += gridDim.x * RED_THREADS) {
        const size_t e = g.index(i);
        f32x4 w[10];
#pragma unroll
        for (int m = 0; m < 10; m++) w[m] = load_group<S>(mom, e + (size_t)m * g.T, L.rscale[m]);
#pragma unroll
        for (int m = 0; m < 10; m++) v[m] += ((double)w[m].x + (double)w[m].y) + ((double)w[m].z + (double)w[m].w);
    }
    block_sum(v);
    if (threadIdx.x == 0)
        for (int m = 0; m < 10; m++) partial[10 * (size_t)blockIdx.x + m] = v[m];
}

// acc (4 x N, x-fastest, FP64) += (rho, ux, uy, uz) of every node
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_mean_accumulate(const void* mom, Linear L, Patches P, float rho0,
                                                                 double* __restrict__ acc) {
    uint32_t x, y, z;
    size_t i;
    if (!P.at(blockIdx.x * RED_THREADS + threadIdx.x, L, x, y, z, i)) return;
    const size_t e = L.at(x, y, z);
    f32x4 w[4];
    f64x4 s[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
        w[a] = load_group<S>(mom, e + (size_t)a * L.T, L.rscale[a]);
        s[a] = ((const f64x4*)acc)[(size_t)a * L.groups + i];
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        s[0][j] += (double)rho0 + (double)w[0][j];
        for (int a = 1; a < 4; a++) s[a][j] += third((double)w[a][j]);
    }
#pragma unroll
    for (int a = 0; a < 4; a++) ((f64x4*)acc)[(size_t)a * L.groups + i] = s[a];
}

// per-workgroup sums of rho |u - mean u|^2, mean u = acc / count
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_tke_partial(const void* mom, Linear L, Patches P, float rho0,
                                                             const double* __restrict__ acc, double inv_count,
                                                             double* __restrict__ partial) {
    double v[1] = {0.0};
    for (uint32_t t = blockIdx.x * RED_THREADS + threadIdx.x; t < P.n; t += gridDim.x * RED_THREADS) {
        uint32_t x, y, z;
        size_t i;
        if (!P.at(t, L, x, y, z, i)) continue;
        const size_t e = L.at(x, y, z);
        const f32x4 r = load_group<S>(mom, e, L.rscale[0]);
        f64x4 k = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int d = 1; d < 4; d++) {
            const f32x4 u = load_group<S>(mom, e + (size_t)d * L.T, L.rscale[d]);
            const f64x4 m = ((const f64x4*)acc)[(size_t)d * L.groups + i];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double du = third((double)u[j]) - m[j] * inv_count;
                k[j] += du * du;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) v[0] += ((double)rho0 + (double)r[j]) * k[j];
    }
    block_sum(v);
    if (threadIdx.x == 0) partial[blockIdx.x] = v[0];
}

unsigned blocks_for(size_t n) { return (unsigned)((n + RED_THREADS - 1) / RED_THREADS); }

int ensure_mean(mrlbm_ctx* c) {
    if (c->d_mean) return MRLBM_OK;
    HIPCHK(hipMalloc((void**)&c->d_mean, sizeof(double) * 4 * c->N));
    HIPCHK(hipMemsetAsync(c->d_mean, 0, sizeof(double) * 4 * c->N, c->stream));
    c->device_bytes += (double)(sizeof(double) * 4 * c->N);
    c->mean_count = 0;
    return MRLBM_OK;
}

}  // namespace

#define MRLBM_DIAG_LAUNCH(KERNEL, GRID, ...)                                                        \
    do {                                                                                            \
        if (c->p.storage == MRLBM_STORE_FP32)                                                       \
            hipLaunchKernelGGL(KERNEL<0>, dim3(GRID), dim3(RED_THREADS), 0, c->stream, __VA_ARGS__); \
        else if (c->p.storage == MRLBM_STORE_FP16)                                                  \
            hipLaunchKernelGGL(KERNEL<1>, dim3(GRID), dim3(RED_THREADS), 0, c->stream, __VA_ARGS__); \
        else                                                                                        \
            hipLaunchKernelGGL(KERNEL<2>, dim3(GRID), dim3(RED_THREADS), 0, c->stream, __VA_ARGS__); \
        HIPCHK(hipGetLastError());                                                                  \
    } while (0)

extern "C" {

int mrlbm_sample(mrlbm_ctx* c, int n, const int32_t* xyz, double* out) {
    if (!c || n < 0 || (n > 0 && (!xyz || !out))) return fail(MRLBM_EINVAL, "bad argument");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    for (int k = 0; k < n; k++)
        if (xyz[3 * k] < 0 || xyz[3 * k] >= c->p.nx || xyz[3 * k + 1] < 0 || xyz[3 * k + 1] >= c->p.ny ||
            xyz[3 * k + 2] < 0 || xyz[3 * k + 2] >= c->p.nz)
            return fail(MRLBM_EINVAL, "sample point %d (%d,%d,%d) outside the lattice", k, xyz[3 * k], xyz[3 * k + 1],
                        xyz[3 * k + 2]);
    if (n == 0) return MRLBM_OK;
    HIPCHK(hipSetDevice(c->p.device));
    const Linear L = linear_of(c);
    // Points that fit the pinned buffer are read and their values written in
    // place: one launch and one wait instead of two allocations, two copies
    // and two frees (16 points: 63 -> 18 us per call).
    constexpr int IN_PLACE = (int)(SMALL_BYTES / (10 * sizeof(double) + 3 * sizeof(int)));
    if (n <= IN_PLACE) {
        std::lock_guard<std::mutex> lock(c->small_mu);
        if (int rc = small_buffer(c)) return rc;
        double* const h_out = (double*)c->h_small;
        int* const h_xyz = (int*)(h_out + 10 * (size_t)n);
        std::memcpy(h_xyz, xyz, sizeof(int) * 3 * (size_t)n);
        MRLBM_DIAG_LAUNCH(k_sample, blocks_for(n), c->d_mom, L, h_xyz, n, h_out);
        HIPCHK(hipStreamSynchronize(c->stream));
        std::memcpy(out, h_out, sizeof(double) * 10 * (size_t)n);
        return MRLBM_OK;
    }
    int* d_xyz = nullptr;
    double* d_out = nullptr;
    HIPCHK(hipMallocAsync((void**)&d_xyz, sizeof(int) * 3 * (size_t)n, c->stream));
    HIPCHK(hipMallocAsync((void**)&d_out, sizeof(double) * 10 * (size_t)n, c->stream));
    HIPCHK(hipMemcpyAsync(d_xyz, xyz, sizeof(int) * 3 * (size_t)n, hipMemcpyHostToDevice, c->stream));
    MRLBM_DIAG_LAUNCH(k_sample, blocks_for(n), c->d_mom, L, d_xyz, n, d_out);
    HIPCHK(hipMemcpyAsync(out, d_out, sizeof(double) * 10 * (size_t)n, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipFreeAsync(d_xyz, c->stream));
    HIPCHK(hipFreeAsync(d_out, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    return MRLBM_OK;
}

int mrlbm_moment_means(mrlbm_ctx* c, double out[10]) {
    if (!c || !out) return fail(MRLBM_EINVAL, "null argument");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    HIPCHK(hipSetDevice(c->p.device));
    std::lock_guard<std::mutex> lock(c->small_mu);
    if (int rc = small_buffer(c)) return rc;
    const BlockGroups g = block_groups((size_t)c->ntiles, c->T);
    const int nb = red_blocks(g.n);
    MRLBM_DIAG_LAUNCH(k_moment_sums, nb, c->d_mom, g, linear_of(c), c->d_partial);
    Divisors<10> div;
    for (double& d : div.d) d = (double)c->N;
    HIPCHK(launch_fold<10>(c->d_partial, nb, (double*)c->h_small, div, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    std::memcpy(out, c->h_small, sizeof(double) * 10);
    return MRLBM_OK;
}

int mrlbm_mean_flow_reset(mrlbm_ctx* c) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    HIPCHK(hipSetDevice(c->p.device));
    if (c->d_mean) HIPCHK(hipMemsetAsync(c->d_mean, 0, sizeof(double) * 4 * c->N, c->stream));
    c->mean_count = 0;
    return MRLBM_OK;
}

int mrlbm_mean_flow_accumulate(mrlbm_ctx* c) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    HIPCHK(hipSetDevice(c->p.device));
    int rc = ensure_mean(c);
    if (rc) return rc;
    const Patches P = patches_of(c);
    MRLBM_DIAG_LAUNCH(k_mean_accumulate, blocks_for(P.n), c->d_mom, linear_of(c), P, (float)c->p.rho0, c->d_mean);
    c->mean_count++;
    return MRLBM_OK;
}

int mrlbm_mean_flow_read(mrlbm_ctx* c, double* out, int64_t* count) {
    if (!c || !out || !count) return fail(MRLBM_EINVAL, "null argument");
    if (!c->d_mean || c->mean_count == 0) return fail(MRLBM_ESTATE, "no mean-flow samples accumulated");
    const int rc = read_scaled(c, c->d_mean, 4 * c->N, 1.0 / (double)c->mean_count, out);
    if (rc) return rc;
    *count = c->mean_count;
    return MRLBM_OK;
}

int mrlbm_turbulent_ke(mrlbm_ctx* c, double* tke) {
    if (!c || !tke) return fail(MRLBM_EINVAL, "null argument");
    if (!c->d_mean || c->mean_count == 0) return fail(MRLBM_ESTATE, "no mean-flow samples accumulated");
    HIPCHK(hipSetDevice(c->p.device));
    std::lock_guard<std::mutex> lock(c->small_mu);
    if (int rc = small_buffer(c)) return rc;
    const Patches P = patches_of(c);
    const int nb = red_blocks(P.n);
    MRLBM_DIAG_LAUNCH(k_tke_partial, nb, c->d_mom, linear_of(c), P, (float)c->p.rho0, c->d_mean,
                      1.0 / (double)c->mean_count, c->d_partial);
    // the kernel sums rho |u - mean u|^2, twice the energy
    HIPCHK(launch_fold<1>(c->d_partial, nb, (double*)c->h_small, {{2.0 * (double)c->N}}, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    *tke = *(const double*)c->h_small;
    return MRLBM_OK;
}

}  // extern "C"
