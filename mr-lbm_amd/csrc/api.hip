// C ABI of the library (include/mrlbm.h): context ownership, node map,
// initial state, step loop, read-back, reductions, checkpoint and VTK.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/mrlbm.h"
#include "bc_classes.h"
#include "context.h"
#include "init_moments.h"
#include "kernels.h"
#include "linear.h"
#include "transfer.h"

using namespace mrlbm;

namespace mrlbm {

thread_local std::string g_err;

int fail(int code, const char* fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

size_t storage_bytes(int storage) { return storage == MRLBM_STORE_FP32 ? 4 : 2; }

// host-side storage conversion (round to nearest even; the kernels round
// stochastically)
uint16_t to_half(double v) { return __builtin_bit_cast(uint16_t, (_Float16)(float)v); }
uint16_t to_bf16(double v) {
    const float f = (float)v;
    uint32_t u;
    std::memcpy(&u, &f, 4);
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

int small_buffer(mrlbm_ctx* c) {
    if (c->h_small) return MRLBM_OK;
    const hipError_t e = hipHostMalloc((void**)&c->h_small, SMALL_BYTES, hipHostMallocDefault);
    if (e != hipSuccess) {
        c->h_small = nullptr;
        return fail(MRLBM_ENOMEM, "pinned result buffer: %s", hipGetErrorString(e));
    }
    return MRLBM_OK;
}

}  // namespace mrlbm

extern "C" {

const char* mrlbm_last_error(void) { return g_err.c_str(); }

int mrlbm_destroy(mrlbm_ctx* c) {
    if (!c) return MRLBM_OK;
    if (c->batch) mrlbm_batch_remove(c->batch, c);
    hipSetDevice(c->p.device);
    if (c->stream) hipStreamSynchronize(c->stream);
    hipFree(c->d_mom);
    hipFree(c->d_cls);
    hipFree(c->d_bc);
    hipFree(c->d_tiles);
    hipFree(c->d_mean);
    for (int s = 0; s < 2; s++)
        hipFree(c->d_gbase[s]);
    hipFree(c->d_partial);
    if (c->h_small) hipHostFree(c->h_small);
    hipFree(c->d_uprev);
    if (c->ev0) hipEventDestroy(c->ev0);
    if (c->ev1) hipEventDestroy(c->ev1);
    if (c->stream) hipStreamDestroy(c->stream);
    delete c;
    count_lattices(-1);
    return MRLBM_OK;
}

int mrlbm_create(const mrlbm_params* pp, mrlbm_ctx** out) {
    if (!pp || !out) return fail(MRLBM_EINVAL, "null argument");
    *out = nullptr;
    const mrlbm_params& p = *pp;
    if (p.q != 19 && p.q != 27) return fail(MRLBM_EINVAL, "q must be 19 or 27 (got %d)", p.q);
    if (p.nx <= 0 || p.ny <= 0 || p.nz <= 0) return fail(MRLBM_EINVAL, "lattice extents must be positive");
    if (p.nx >= (1 << 24)) return fail(MRLBM_EINVAL, "nx must be below 2^24");  // 24-bit node-key multiply
    if (!(p.tau > 0.5)) return fail(MRLBM_EINVAL, "tau must exceed 0.5 (got %g)", p.tau);
    if (p.storage != MRLBM_STORE_FP32 && p.storage != MRLBM_STORE_FP16 && p.storage != MRLBM_STORE_BF16)
        return fail(MRLBM_EINVAL, "unknown storage precision %d", p.storage);
    if (p.kernel != MRLBM_KERNEL_AUTO && p.kernel != MRLBM_KERNEL_TILE && p.kernel != MRLBM_KERNEL_COLUMN)
        return fail(MRLBM_EINVAL, "unknown kernel family %d", p.kernel);
    int bx = p.bx, by = p.by, bz = p.bz;
    int kernel = p.kernel;
    if (bx == 0 && by == 0 && bz == 0) {
        // default: the fastest measured tile that divides the lattice, or for
        // the column kernel the longest segment that does. FP32 D3Q19 is
        // HBM-bound, and 16x8x8 tiles move 105 instead of 110 B per update
        // (256^3 TGV 54.9 -> 57.7 GLUPS, cavity 50.9 -> 51.3); the 16-bit
        // storages and D3Q27 are bound by instruction issue and latency,
        // which the 1024-thread tiles' two workgroups per CU hide worse
        // (FP16 TGV 74.9 -> 68.0 GLUPS), so they keep 8x8x8.
        const bool big = p.q == 19 && p.storage == MRLBM_STORE_FP32;
        const int cand[4][3] = {{16, 8, 8}, {8, 8, 8}, {16, 16, 32}, {16, 16, 64}};
        for (int c = big ? 0 : 1; c < 4; c++) {
            const bool col = cand[c][0] * cand[c][1] == 256;
            if (kernel != MRLBM_KERNEL_COLUMN && col) continue;
            if (kernel == MRLBM_KERNEL_COLUMN && !col) continue;
            if (p.nx % cand[c][0] == 0 && p.ny % cand[c][1] == 0 && p.nz % cand[c][2] == 0) {
                bx = cand[c][0];
                by = cand[c][1];
                bz = cand[c][2];
                break;
            }
        }
        if (bx == 0) return fail(MRLBM_EINVAL, "no built tile shape divides %dx%dx%d", p.nx, p.ny, p.nz);
    }
    if (kernel == MRLBM_KERNEL_AUTO) kernel = (bx * by == 256 && bz > 8) ? MRLBM_KERNEL_COLUMN : MRLBM_KERNEL_TILE;
    if (kernel == MRLBM_KERNEL_TILE && !tile_shape_supported(p.q, bx, by, bz, p.storage))
        return fail(MRLBM_EINVAL, "tile shape %dx%dx%d not built for q=%d storage=%d", bx, by, bz, p.q, p.storage);
    if (kernel == MRLBM_KERNEL_COLUMN && !column_shape_supported(p.q, bx, by, bz, p.storage))
        return fail(MRLBM_EINVAL, "column shape %dx%dx%d not built for q=%d storage=%d", bx, by, bz, p.q, p.storage);
    if (p.nx % bx || p.ny % by || p.nz % bz)
        return fail(MRLBM_EINVAL, "lattice %dx%dx%d is not a multiple of the tile %dx%dx%d", p.nx, p.ny, p.nz, bx, by,
                    bz);
    int ndev = 0;
    HIPCHK(hipGetDeviceCount(&ndev));
    if (p.device < 0 || p.device >= ndev) return fail(MRLBM_EINVAL, "device %d not present", p.device);
    HIPCHK(hipSetDevice(p.device));
    // set-up of the device's scratch array for mrlbm_reduce_checked_noalloc
    // (once per device: the symbol lookup is not an allocation)
    if (int rc0 = noalloc_scratch_setup(p.device, nullptr)) return rc0;

    mrlbm_ctx* c = new mrlbm_ctx();
    count_lattices(1);
    c->p = p;
    if (c->p.rho0 == 0.0) c->p.rho0 = 1.0;
    c->p.bx = c->bx = bx;
    c->p.by = c->by = by;
    c->p.bz = c->bz = bz;
    c->p.kernel = kernel;
    c->T = bx * by * bz;
    c->ntx = p.nx / bx;
    c->nty = p.ny / by;
    c->ntz = p.nz / bz;
    c->ntiles = c->ntx * c->nty * c->ntz;
    c->qf = p.q == 19 ? 5 : 9;
    c->N = (size_t)p.nx * p.ny * p.nz;
    // storage scales (powers of two), the same constants the step kernels use
    static_assert(MRLBM_STORE_FP16 == 1 && MRLBM_STORE_BF16 == 2, "storage codes");
    for (int m = 0; m < 10; m++) {
        const float s = store_scale(p.storage, m);
        c->mscale[m] = s;
        c->mrscale[m] = 1.0f / s;
    }

    auto alloc = [&](void** ptr, size_t bytes) -> int {
        hipError_t e = hipMalloc(ptr, bytes);
        if (e != hipSuccess) {
            *ptr = nullptr;
            return fail(MRLBM_ENOMEM, "hipMalloc(%zu bytes) failed: %s", bytes, hipGetErrorString(e));
        }
        c->device_bytes += (double)bytes;
        return MRLBM_OK;
    };
    int rc;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
        mrlbm_destroy(c);
        return fail(MRLBM_EHIP, "hipStreamCreate failed");
    }
    if ((rc = alloc(&c->d_mom, c->N * 10 * storage_bytes(p.storage)))) {
        mrlbm_destroy(c);
        return rc;
    }
    c->face_elems[0] = c->face_elems[1] = (size_t)by * bz * c->qf * c->ntiles;
    c->face_elems[2] = c->face_elems[3] = (size_t)bx * bz * c->qf * c->ntiles;
    c->face_elems[4] = c->face_elems[5] = (size_t)bx * by * c->qf * c->ntiles;
    for (int s = 0; s < 2; s++) {
        size_t set = 0;
        for (int f = 0; f < 6; f++) set += c->face_elems[f];
        if ((rc = alloc((void**)&c->d_gbase[s], set * sizeof(float)))) {
            mrlbm_destroy(c);
            return rc;
        }
        size_t o = 0;
        for (int f = 0; f < 6; f++) {
            c->d_ghost[s][f] = c->d_gbase[s] + o;
            o += c->face_elems[f];
        }
    }
    if ((rc = alloc((void**)&c->d_partial, sizeof(double) * 10 * RED_BLOCKS_MAX))) {
        mrlbm_destroy(c);
        return rc;
    }
    if (hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        mrlbm_destroy(c);
        return fail(MRLBM_EHIP, "hipEventCreate failed");
    }
    *out = c;
    return MRLBM_OK;
}

int mrlbm_set_bc_velocity(mrlbm_ctx* c, int k, double ux, double uy, double uz) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    if (k < 0 || k > 3) return fail(MRLBM_EINVAL, "wall-velocity index %d outside 0..3", k);
    c->bc_vel[k][0] = ux;
    c->bc_vel[k][1] = uy;
    c->bc_vel[k][2] = uz;
    return MRLBM_OK;
}

int mrlbm_set_node_types(mrlbm_ctx* c, const uint32_t* types) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    HIPCHK(hipSetDevice(c->p.device));
    BcClassTable tab;
    std::string err = build_class_table(c->p.q, 1.0 / c->p.tau, c->bc_vel, types, c->N, tab);
    if (!err.empty()) return fail(MRLBM_EINVAL, "%s", err.c_str());
    HIPCHK(hipStreamSynchronize(c->stream));
    hipFree(c->d_cls);
    hipFree(c->d_bc);
    c->d_cls = nullptr;
    c->d_bc = nullptr;
    c->bc_bytes = 0;
    c->has_bc = tab.has_bc;
    c->has_solid = tab.has_solid;
    c->n_classes = (int)tab.keys.size() - 1;
    c->version++;
    c->cls_version++;
    if (!c->has_bc) return build_tile_list(c);
    std::vector<uint8_t> blk(c->N);
    const int nx = c->p.nx, ny = c->p.ny, nz = c->p.nz;
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < ny; y++)
            for (int x = 0; x < nx; x++) blk[c->node_index(x, y, z)] = tab.class_of[x + (size_t)nx * (y + (size_t)ny * z)];
    HIPCHK(hipMalloc((void**)&c->d_cls, c->N));
    HIPCHK(hipMalloc((void**)&c->d_bc, tab.table.size() * sizeof(float)));
    c->bc_bytes = tab.table.size() * sizeof(float);
    HIPCHK(hipMemcpy(c->d_cls, blk.data(), c->N, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(c->d_bc, tab.table.data(), tab.table.size() * sizeof(float), hipMemcpyHostToDevice));
    return build_tile_list(c);
}

}  // extern "C"

namespace {

// One stored moment (index m, stored convention) -> its storage word
uint32_t encode_value(const mrlbm_ctx* c, int m, double x) {
    const double v = x * c->mscale[m];
    if (c->p.storage == MRLBM_STORE_FP32) {
        const float f = (float)v;
        uint32_t u;
        std::memcpy(&u, &f, 4);
        return u;
    }
    return c->p.storage == MRLBM_STORE_FP16 ? to_half(v) : to_bf16(v);
}

// Both ghost sets from the stored moments; the lattice restarts at step 0.
int ghosts_from_moments(mrlbm_ctx* c) {
    StepArgs a = c->args();
    for (int s = 0; s < 2; s++) {
        if (c->p.kernel == MRLBM_KERNEL_COLUMN)
            HIPCHK(launch_init_ghosts_column(c->p.q, c->bx, c->by, c->bz, c->p.storage, a, c->d_ghost[s], c->ntiles,
                                             c->stream));
        else
            HIPCHK(launch_init_ghosts(c->p.q, c->bx, c->by, c->bz, c->p.storage, a, c->d_ghost[s], c->ntiles,
                                      c->stream));
    }
    HIPCHK(hipStreamSynchronize(c->stream));
    c->cur = 0;
    c->step = 0;
    c->initialised = true;
    c->version++;
    return MRLBM_OK;
}

int check_mode(int mode) {
    if (mode != MRLBM_INIT_EQUILIBRIUM && mode != MRLBM_INIT_REFERENCE)
        return fail(MRLBM_EINVAL, "unknown second-moment mode %d", mode);
    return MRLBM_OK;
}

}  // namespace

extern "C" {

int mrlbm_init_fields(mrlbm_ctx* c, const double* rho, const double* ux, const double* uy, const double* uz,
                      int mode) {
    if (!c || !rho || !ux || !uy || !uz) return fail(MRLBM_EINVAL, "null argument");
    int rc = check_mode(mode);
    if (!rc) rc = write_fields_linear(c, mode, rho, ux, uy, uz);
    return rc ? rc : ghosts_from_moments(c);
}

int mrlbm_init_uniform(mrlbm_ctx* c, double rho, double ux, double uy, double uz, int mode) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    int rc = check_mode(mode);
    if (rc) return rc;
    if (!(rho > 0)) return fail(MRLBM_EINVAL, "non-positive density");
    // one node's stored moments, encoded once and filled on the device
    double m[10];
    node_moments(c->p.q, mode, c->p.rho0, rho, ux, uy, uz, m);
    uint32_t enc[10];
    for (int k = 0; k < 10; k++) enc[k] = encode_value(c, k, m[k]);
    HIPCHK(hipSetDevice(c->p.device));
    if ((rc = fill_uniform_moments(c, enc))) return rc;
    return ghosts_from_moments(c);
}

int mrlbm_init_taylor_green(mrlbm_ctx* c, double u0, int mode) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    int rc = check_mode(mode);
    if (!rc) rc = write_taylor_green(c, u0, mode);
    return rc ? rc : ghosts_from_moments(c);
}

static int do_steps(mrlbm_ctx* c, int nsteps) {
    const bool split = c->p.kernel == MRLBM_KERNEL_TILE && c->has_bc && c->d_tiles;
    const bool mixed = split && mixed_launch_supported(c->p.q, c->bx, c->by, c->bz, c->p.storage);
    for (int s = 0; s < nsteps; s++) {
        StepArgs a = c->args();
        hipError_t e;
        if (c->p.kernel == MRLBM_KERNEL_COLUMN) {
            e = launch_step_column(c->p.q, c->bx, c->by, c->bz, c->has_bc, c->p.storage, a, c->ntiles, c->stream);
        } else if (split && mixed) {
            // one launch: the all-bulk tiles with the light body, the rest
            // with the boundary body
            e = launch_step_tile_mixed(c->p.q, c->bx, c->by, c->bz, c->p.storage, a, c->d_tiles, c->ntiles,
                                       c->n_bulk_tiles, c->stream);
        } else if (split) {
            // all-bulk tiles with the light body, the rest with boundaries;
            // both read the same ghost set and write disjoint data
            e = launch_step_tile(c->p.q, c->bx, c->by, c->bz, false, c->p.storage, a, c->d_tiles, c->n_bulk_tiles,
                                 c->stream);
            if (e == hipSuccess)
                e = launch_step_tile(c->p.q, c->bx, c->by, c->bz, true, c->p.storage, a, c->d_tiles + c->n_bulk_tiles,
                                     c->ntiles - c->n_bulk_tiles, c->stream);
        } else {
            e = launch_step_tile(c->p.q, c->bx, c->by, c->bz, c->has_bc, c->p.storage, a, nullptr, c->ntiles,
                                 c->stream);
        }
        if (e != hipSuccess) return fail(MRLBM_EHIP, "step launch failed: %s", hipGetErrorString(e));
        c->cur = 1 - c->cur;
        c->step++;
    }
    return MRLBM_OK;
}

int mrlbm_step(mrlbm_ctx* c, int nsteps) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    if (c->batch) return fail(MRLBM_ESTATE, "lattice is stepped by its batch (mrlbm_batch_step)");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    if (nsteps < 0) return fail(MRLBM_EINVAL, "negative step count");
    HIPCHK(hipSetDevice(c->p.device));
    return do_steps(c, nsteps);
}

int mrlbm_time_steps(mrlbm_ctx* c, int nsteps, double* ms) {
    if (!c || !ms) return fail(MRLBM_EINVAL, "null argument");
    if (c->batch) return fail(MRLBM_ESTATE, "lattice is stepped by its batch (mrlbm_batch_time_steps)");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    HIPCHK(hipSetDevice(c->p.device));
    HIPCHK(hipEventRecord(c->ev0, c->stream));
    int rc = do_steps(c, nsteps);
    if (rc) return rc;
    HIPCHK(hipEventRecord(c->ev1, c->stream));
    HIPCHK(hipEventSynchronize(c->ev1));
    float f = 0;
    HIPCHK(hipEventElapsedTime(&f, c->ev0, c->ev1));
    *ms = f;
    return MRLBM_OK;
}

int mrlbm_synchronize(mrlbm_ctx* c) {
    if (!c) return fail(MRLBM_EINVAL, "null context");
    HIPCHK(hipSetDevice(c->p.device));
    HIPCHK(hipStreamSynchronize(c->stream));
    return MRLBM_OK;
}

int mrlbm_read_moments(mrlbm_ctx* c, double* out) {
    if (!c || !out) return fail(MRLBM_EINVAL, "null argument");
    return read_moments_linear(c, out);
}

int mrlbm_read_macroscopic(mrlbm_ctx* c, double rho0, double* out) {
    if (!c || !out) return fail(MRLBM_EINVAL, "null argument");
    double* const plane[4] = {out, out + c->N, out + 2 * c->N, out + 3 * c->N};
    return read_macroscopic_linear(c, rho0, plane);
}

int mrlbm_read_fields(mrlbm_ctx* c, double rho0, double* rho, double* ux, double* uy, double* uz) {
    if (!c || !rho || !ux || !uy || !uz) return fail(MRLBM_EINVAL, "null argument");
    double* const plane[4] = {rho, ux, uy, uz};
    return read_macroscopic_linear(c, rho0, plane);
}

int mrlbm_write_moments(mrlbm_ctx* c, const double* in) {
    if (!c || !in) return fail(MRLBM_EINVAL, "null argument");
    const int rc = write_moments_linear(c, in);
    return rc ? rc : ghosts_from_moments(c);
}

int mrlbm_reduce_checked(mrlbm_ctx* c, double* mass, double* ke, int64_t* nonfinite) {
    if (!c || !mass || !ke || !nonfinite) return fail(MRLBM_EINVAL, "null argument");
    HIPCHK(hipSetDevice(c->p.device));
    std::lock_guard<std::mutex> lock(c->small_mu);
    if (int rc = small_buffer(c)) return rc;
    double* const h = (double*)c->h_small;
    HIPCHK(launch_reduce(c->p.storage, c->d_mom, c->ntiles, c->T, (float)c->p.rho0, c->mrscale[0], c->mrscale[1],
                         c->d_partial, h, c->stream, (double)c->N));
    HIPCHK(hipStreamSynchronize(c->stream));
    *mass = h[0];
    *ke = h[1];
    *nonfinite = (int64_t)h[2];
    return MRLBM_OK;
}

int mrlbm_reduce(mrlbm_ctx* c, double* mass, double* ke) {
    int64_t bad;
    return mrlbm_reduce_checked(c, mass, ke, &bad);
}

int mrlbm_velocity_residual(mrlbm_ctx* c, double* residual) {
    if (!c || !residual) return fail(MRLBM_EINVAL, "null argument");
    if (!c->initialised) return fail(MRLBM_ESTATE, "lattice not initialised");
    HIPCHK(hipSetDevice(c->p.device));
    std::lock_guard<std::mutex> lock(c->small_mu);
    // before the reference: a call that fails here leaves the next one the first
    if (int rc = small_buffer(c)) return rc;
    const bool first = c->d_uprev == nullptr;
    if (first) {
        const size_t bytes = sizeof(float) * 3 * c->N;
        if (hipMalloc((void**)&c->d_uprev, bytes) != hipSuccess) {
            c->d_uprev = nullptr;
            return fail(MRLBM_ENOMEM, "hipMalloc(%zu bytes) for the residual reference failed", bytes);
        }
        c->device_bytes += (double)bytes;
        HIPCHK(hipMemsetAsync(c->d_uprev, 0, bytes, c->stream));
    }
    double* const h = (double*)c->h_small;
    HIPCHK(launch_residual(c->p.storage, c->d_mom, c->d_uprev, c->ntiles, c->T, c->mrscale[1], c->d_partial, h,
                           c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    *residual = first ? -1.0 : (h[1] > 0.0 ? std::sqrt(h[0] / h[1]) : (h[0] > 0.0 ? INFINITY : 0.0));
    return MRLBM_OK;
}

int mrlbm_get_info(mrlbm_ctx* c, mrlbm_info* o) {
    if (!c || !o) return fail(MRLBM_EINVAL, "null argument");
    o->nx = c->p.nx;
    o->ny = c->p.ny;
    o->nz = c->p.nz;
    o->q = c->p.q;
    o->bx = c->bx;
    o->by = c->by;
    o->bz = c->bz;
    o->storage = c->p.storage;
    o->kernel = c->p.kernel;
    o->step = c->step;
    o->n_bc_classes = c->n_classes;
    o->has_solid = c->has_solid;
    o->bytes_per_lu = c->bytes_per_lu();
    o->device_bytes = c->device_bytes;
    return MRLBM_OK;
}

int mrlbm_bc_class_info(int q, uint32_t node_type, double omega, const double u[3], uint32_t* known,
                        double* ainv49) {
    if (!u || !known || !ainv49) return fail(MRLBM_EINVAL, "null argument");
    if (q != 19 && q != 27) return fail(MRLBM_EINVAL, "q must be 19 or 27");
    *known = known_mask(q, node_type & 0xFFu);
    if (!build_bc_inverse(q, *known, omega, u, ainv49, nullptr, closure_lattice(q, node_type & 0xFFu)))
        return fail(MRLBM_ENUMERIC, "singular boundary system");
    return MRLBM_OK;
}

}  // extern "C"
