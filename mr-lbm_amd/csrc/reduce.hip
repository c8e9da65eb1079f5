// FP64 lattice reductions: sum of (rho - RHO_0) and of rho |u|^2 / 2 over
// all nodes (solid nodes included, as the reference's sumReductionThread_rho
// / sumReductionThread_KE do, src/reduction.cu:99-155), with a count of
// non-finite nodes, and the velocity convergence residual. The reference sums
// in FP32 with repeated block passes; here each thread accumulates in FP64
// over groups of four nodes, the workgroup sums by lane shuffles, and a single
// workgroup folds the partials in a fixed order, so the result is
// deterministic for a given lattice. Bound: memory (the moment planes read
// once; the index of a group is shifts and a multiply, no division). FP32
// 192x160x128: reduction 16.7 -> 11.9 us, residual 39.4 -> 25.1 us, their
// folds 6 -> 4 us.
#include <mutex>
#include <vector>

#include "context.h"
#include "linear.h"

namespace mrlbm {

namespace {

// Exponent all ones: infinity or NaN.
__device__ __forceinline__ bool finite32(float x) { return (__float_as_uint(x) & 0x7F800000u) != 0x7F800000u; }

// Per workgroup: sums of (rho - RHO_0) and rho |3u|^2, and the number of
// nodes whose rho - RHO_0 or u is not finite (any such node also makes the
// sums non-finite; the count says how many). partial[3 b + 0..2].
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_reduce_partial(const void* mom, BlockGroups g, float rho0, float rs0,
                                                               float rs1, double* partial) {
    double v[3] = {0.0, 0.0, 0.0};
    for (uint32_t i = blockIdx.x * RED_THREADS + threadIdx.x; i < g.n; i += gridDim.x * RED_THREADS) {
        const size_t e = g.index(i);
        const f32x4 r = load_group<S>(mom, e, rs0), x = load_group<S>(mom, e + g.T, rs1),
                    y = load_group<S>(mom, e + 2 * (size_t)g.T, rs1), z = load_group<S>(mom, e + 3 * (size_t)g.T, rs1);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const double dr = r[j], ux = x[j], uy = y[j], uz = z[j];
            v[0] += dr;
            v[1] += ((double)rho0 + dr) * (ux * ux + uy * uy + uz * uz);
            v[2] += finite32(r[j]) && finite32(x[j]) && finite32(y[j]) && finite32(z[j]) ? 0.0 : 1.0;
        }
    }
    block_sum(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; k++) partial[3 * blockIdx.x + k] = v[k];
}

template <int K>
__global__ __launch_bounds__(RED_THREADS) void k_fold(const double* partial, int n, double* out, Divisors<K> div) {
    double v[K] = {};
    for (int j = threadIdx.x; j < n; j += RED_THREADS)
        for (int k = 0; k < K; k++) v[k] += partial[K * j + k];
    block_sum(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < K; k++) out[k] = v[k] / div.d[k];
}

// Convergence residual: per workgroup, sums over nodes of |u - u_prev|^2 and
// of |u|^2 (u from the stored moments, u_prev a saved FP32 copy, 3 planes of
// N values in block layout); u_prev is then overwritten with u.
template <int S>
__global__ __launch_bounds__(RED_THREADS) void k_residual_partial(const void* mom, float* uprev, BlockGroups g,
                                                                  float rs1, double* partial) {
    double v[2] = {0.0, 0.0};
    for (uint32_t i = blockIdx.x * RED_THREADS + threadIdx.x; i < g.n; i += gridDim.x * RED_THREADS) {
        const size_t e = g.index(i);
        f32x4 u[3], p[3];
#pragma unroll
        for (int a = 0; a < 3; a++) {
            u[a] = load_group<S>(mom, e + (size_t)(1 + a) * g.T, rs1) * (1.0f / 3.0f);
            p[a] = __builtin_nontemporal_load((const f32x4*)uprev + (size_t)a * g.n + i);
        }
#pragma unroll
        for (int a = 0; a < 3; a++) {
            __builtin_nontemporal_store(u[a], (f32x4*)uprev + (size_t)a * g.n + i);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const double d = (double)u[a][j] - (double)p[a][j];
                v[0] += d * d;
                v[1] += (double)u[a][j] * (double)u[a][j];
            }
        }
    }
    block_sum(v);
    if (threadIdx.x == 0)
        for (int k = 0; k < 2; k++) partial[2 * blockIdx.x + k] = v[k];
}

}  // namespace

template <int K>
hipError_t launch_fold(const double* partial, int n, double* out, const Divisors<K>& div, hipStream_t s) {
    hipLaunchKernelGGL(k_fold<K>, dim3(1), dim3(RED_THREADS), 0, s, partial, n, out, div);
    return hipGetLastError();
}
template hipError_t launch_fold<1>(const double*, int, double*, const Divisors<1>&, hipStream_t);
template hipError_t launch_fold<10>(const double*, int, double*, const Divisors<10>&, hipStream_t);

hipError_t launch_reduce(int storage, const void* mom, size_t ntiles, int tile_nodes, float rho0, float rs0, float rs1,
                         double* partial, double* out3, hipStream_t s, double n_nodes) {
    const BlockGroups g = block_groups(ntiles, tile_nodes);
    const int nb = red_blocks(g.n);
    const dim3 grid(nb), block(RED_THREADS);
    if (storage == 0)
        hipLaunchKernelGGL(k_reduce_partial<0>, grid, block, 0, s, mom, g, rho0, rs0, rs1, partial);
    else if (storage == 1)
        hipLaunchKernelGGL(k_reduce_partial<1>, grid, block, 0, s, mom, g, rho0, rs0, rs1, partial);
    else if (storage == 2)
        hipLaunchKernelGGL(k_reduce_partial<2>, grid, block, 0, s, mom, g, rho0, rs0, rs1, partial);
    else
        return hipErrorInvalidValue;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // the kernel sums rho |3u|^2 = 18 (rho |u|^2 / 2)
    return launch_fold<3>(partial, nb, out3, {{n_nodes, 18.0 * n_nodes, 1.0}}, s);
}

hipError_t launch_residual(int storage, const void* mom, float* uprev, size_t ntiles, int tile_nodes, float rs1,
                           double* partial, double* out2, hipStream_t s) {
    const BlockGroups g = block_groups(ntiles, tile_nodes);
    const int nb = red_blocks(g.n);
    const dim3 grid(nb), block(RED_THREADS);
    if (storage == 0)
        hipLaunchKernelGGL(k_residual_partial<0>, grid, block, 0, s, mom, uprev, g, rs1, partial);
    else if (storage == 1)
        hipLaunchKernelGGL(k_residual_partial<1>, grid, block, 0, s, mom, uprev, g, rs1, partial);
    else if (storage == 2)
        hipLaunchKernelGGL(k_residual_partial<2>, grid, block, 0, s, mom, uprev, g, rs1, partial);
    else
        return hipErrorInvalidValue;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_fold<2>(partial, nb, out2, {{1.0, 1.0}}, s);
}

// ---------------------------------------------------------------------------
// Allocation-free checked reduction (mrlbm_reduce_checked_noalloc). The
// partial sums live in a file-scope device array, one copy per device for
// the life of the process, instead of the context's partial buffer; the
// kernels and the block count are those of mrlbm_reduce_checked, so the
// result is the same bit for bit. In host code `scratch` names a host-side
// stand-in: kernels get the device address that hipGetSymbolAddress returns
// for the current device, looked up once per device and kept.
static __device__ __align__(256) double scratch[3 * RED_BLOCKS_MAX];  // 1024 partial triples, 24 KiB

namespace {
std::mutex g_scratch_mu;
std::vector<double*> g_scratch;  // per device: device address of `scratch`
}  // namespace

int noalloc_scratch_setup(int device, double** out) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (device < 0) return fail(MRLBM_EINVAL, "device %d", device);
    if ((int)g_scratch.size() <= device) g_scratch.resize((size_t)device + 1, nullptr);
    if (!g_scratch[device]) {
        int cur = -1;
        HIPCHK(hipGetDevice(&cur));
        if (cur != device) return fail(MRLBM_EHIP, "scratch set-up for device %d while device %d is current", device, cur);
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(MRLBM_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
        g_scratch[device] = (double*)p;
    }
    if (out) *out = g_scratch[device];
    return MRLBM_OK;
}

}  // namespace mrlbm

extern "C" int mrlbm_reduce_checked_noalloc(mrlbm_ctx* c, double* d_out3) {
    using namespace mrlbm;
    if (!c || !d_out3) return fail(MRLBM_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->p.device));
    hipPointerAttribute_t at{};
    if (hipPointerGetAttributes(&at, d_out3) != hipSuccess || at.type != hipMemoryTypeDevice || at.device != c->p.device) {
        (void)hipGetLastError();  // clear the query's error state
        return fail(MRLBM_EINVAL, "d_out3 must be device memory on device %d", c->p.device);
    }
    double* part = nullptr;
    const int rc = noalloc_scratch_setup(c->p.device, &part);
    if (rc) return rc;
    HIPCHK(launch_reduce(c->p.storage, c->d_mom, c->ntiles, c->T, (float)c->p.rho0, c->mrscale[0], c->mrscale[1], part,
                         d_out3, c->stream, (double)c->N));
    return MRLBM_OK;
}
