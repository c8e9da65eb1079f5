// Whole fields between the caller's host arrays and HBM: read-back of the
// stored moments and of the mean flow, initial states and rewritten moments.
//
// The device does the layout and the format: kernels gather the block-major
// moments into x-fastest order (or scatter them from it), decode or encode
// the storage words and evaluate the stored moments of an initial state, and
// read or write pinned host memory directly. The host only moves contiguous
// runs between the caller's (pageable) arrays and the pinned slots. Bound:
// PCIe (57 GB/s pinned on MI355X) and the host's own memory, so moments
// cross PCIe as FP32 (every stored value is exact in FP32) and are widened
// to FP64 as they are copied out.
// Decoding, transposing and index arithmetic on one host thread took
// 0.95 s for the moments of 256^3 FP32 (1.34 GB as FP64; now 26 ms) and
// 1.76 s for the Taylor-Green state (now about a millisecond).
#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

#include "context.h"
#include "init_moments.h"
#include "linear.h"
#include "transfer.h"

using namespace mrlbm;

namespace {

constexpr int THREADS = 256;
// A slot is what one kernel moves; each worker has two, so that the copy of
// one overlaps the transfer of the other. 1 MiB is the smallest size that
// still moves at the PCIe rate (50 GB/s back to back; 256 KiB: 36 GB/s).
constexpr size_t SLOT_BYTES = 1u << 20;
// One core widens 22 GB/s into fresh memory, four 50 GB/s, eight 76 GB/s
// (measured; PCIe delivers 108 GB/s of widened values): more than eight add
// nothing. A worker is worth its thread (60 us to start and join) from about
// three slots on.
constexpr int MAX_WORKERS = 8;
constexpr size_t CHUNKS_PER_WORKER = 3;

int workers_for(size_t chunks) {
    const unsigned hw = std::thread::hardware_concurrency();
    size_t w = chunks / CHUNKS_PER_WORKER;
    if (w > MAX_WORKERS) w = MAX_WORKERS;
    if (hw && w > hw) w = hw;
    return w < 1 ? 1 : (int)w;
}

// f(0) .. f(n - 1), each on a thread of its own (the last on the caller's);
// where no thread can be started the caller runs the rest.
template <typename F>
void run_workers(int n, F&& f) {
    std::thread th[MAX_WORKERS];
    int started = 0;
    try {
        for (; started < n - 1; started++) th[started] = std::thread([&f, started] { f(started); });
    } catch (const std::system_error&) {
    } catch (const std::bad_alloc&) {
    }
    for (int w = started; w < n; w++) f(w);
    for (int w = 0; w < started; w++) th[w].join();
}

// Pinned slots of the process: a call takes what is free and allocates the
// rest, and gives them back; at most two per possible worker stay, for as
// long as any lattice lives (mrlbm_create and mrlbm_destroy count them). A
// fresh slab of 16 MiB costs 0.4 ms to allocate and as much again on its first
// use, a slot by itself about 15 us, and a living lattice's next transfer
// nothing (create, two transfers and destroy of a 96x72x80 lattice: 3.7 ms
// with a slab per call, 2.3 ms; slots in pairs of 2 MiB, past what the runtime
// cuts from its own blocks, 4.8 ms).
struct SlotPool {
    static constexpr size_t KEPT = 2 * MAX_WORKERS;
    std::mutex mu;
    char* kept[KEPT];
    size_t n = 0;
    int lattices = 0;
    hipError_t take(char** p) {
        {
            std::lock_guard<std::mutex> lock(mu);
            if (n) {
                *p = kept[--n];
                return hipSuccess;
            }
        }
        return hipHostMalloc((void**)p, SLOT_BYTES, hipHostMallocPortable);
    }
    void give(char* p) {
        {
            std::lock_guard<std::mutex> lock(mu);
            if (lattices > 0 && n < KEPT) {
                kept[n++] = p;
                return;
            }
        }
        (void)hipHostFree(p);
    }
    void count(int d) {
        size_t m = 0;
        char* drop[KEPT];
        {
            std::lock_guard<std::mutex> lock(mu);
            lattices += d;
            if (lattices == 0) {
                for (m = 0; m < n; m++) drop[m] = kept[m];
                n = 0;
            }
        }
        for (size_t k = 0; k < m; k++) (void)hipHostFree(drop[k]);
    }
};
SlotPool g_slots;

// Pinned slots and their events for one call.
struct Slots {
    char* mem[2 * MAX_WORKERS] = {};
    hipEvent_t ev[2 * MAX_WORKERS] = {};
    int n = 0;
    hipError_t open(int slots) {
        for (; n < slots; n++) {
            hipError_t e = g_slots.take(&mem[n]);
            if (e != hipSuccess) return e;
            if ((e = hipEventCreateWithFlags(&ev[n], hipEventDisableTiming)) != hipSuccess) {
                g_slots.give(mem[n]);
                return e;
            }
        }
        return hipSuccess;
    }
    ~Slots() {
        for (int k = 0; k < n; k++) {
            (void)hipEventDestroy(ev[k]);
            g_slots.give(mem[k]);
        }
    }
    char* at(int k) const { return mem[k]; }
};

// Moves `chunks` chunks through pinned slots, worker w taking w, w + W, ...
// DOWN: launch(c, slot) makes the device fill the slot, take(c, slot) empties
// it on the host; otherwise take fills it and launch makes the device read
// it. Returns when every chunk has arrived and the stream is idle.
template <bool DOWN, typename Launch, typename Take>
int pump(mrlbm_ctx* c, size_t chunks, Launch&& launch, Take&& take) {
    HIPCHK(hipSetDevice(c->p.device));
    if (chunks == 0) return MRLBM_OK;
    const int W = workers_for(chunks);
    Slots slots;
    hipError_t e = slots.open((size_t)(2 * W) < chunks ? 2 * W : (int)chunks);
    if (e != hipSuccess) return fail(MRLBM_ENOMEM, "pinned staging memory: %s", hipGetErrorString(e));
    std::atomic<int> err{(int)hipSuccess};
    auto worker = [&](int w) {
        auto ok = [&](hipError_t r) {
            if (r != hipSuccess) err = (int)r;
            return r == hipSuccess;
        };
        if (!ok(hipSetDevice(c->p.device))) return;
        auto send = [&](size_t k, int s) { return ok(launch(k, slots.at(s))) && ok(hipEventRecord(slots.ev[s], c->stream)); };
        if constexpr (DOWN) {
            size_t ahead = w;
            for (int b = 0; b < 2 && ahead < chunks; b++, ahead += W)
                if (!send(ahead, 2 * w + b)) return;
            for (size_t k = w, b = 0; k < chunks; k += W, b ^= 1) {
                const int s = 2 * w + (int)b;
                if (!ok(hipEventSynchronize(slots.ev[s]))) return;
                take(k, slots.at(s));
                if (ahead < chunks) {
                    if (!send(ahead, s)) return;
                    ahead += W;
                }
            }
        } else {
            size_t n = 0;
            for (size_t k = w; k < chunks; k += W, n++) {
                const int s = 2 * w + (int)(n & 1);
                if (n >= 2 && !ok(hipEventSynchronize(slots.ev[s]))) return;
                take(k, slots.at(s));
                if (!send(k, s)) return;
            }
        }
    };
    run_workers(W, worker);
    // the slots are released below: nothing may still use them
    e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = (hipError_t)err.load();
    if (e != hipSuccess) return fail(MRLBM_EHIP, "field transfer: %s", hipGetErrorString(e));
    return MRLBM_OK;
}

// Moment plane and group of group `i` of a chunk that starts at group j0 of
// plane k0 (a chunk of a small lattice spans planes).
__device__ __forceinline__ void plane_group(const Linear& L, uint32_t i, int& k, uint32_t& j) {
    uint64_t jj = (uint64_t)j + i;
    while (jj >= L.groups) jj -= L.groups, k++;
    j = (uint32_t)jj;
}

// n groups of decoded values in output order, one group per thread: reads
// runs of a tile row, writes whole lines of the pinned slot. PCIe-bound
// (1 MiB in 20 us).
template <int S>
__global__ __launch_bounds__(THREADS) void k_read_linear(const void* mom, Linear L, int k0, uint32_t j0, uint32_t n,
                                                         f32x4* __restrict__ out) {
    using W = Word<S>;
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if (i >= n) return;
    int k = k0;
    uint32_t j = j0;
    plane_group(L, i, k, j);
    const auto w = __builtin_nontemporal_load(
        (const typename W::V*)((const typename W::T*)mom + L.node(j) + (size_t)k * L.T));
    const float rs = L.rscale[k];
    const f32x4 v = {W::dec(w.x, rs), W::dec(w.y, rs), W::dec(w.z, rs), W::dec(w.w, rs)};
    __builtin_nontemporal_store(v, &out[i]);
}

// The reverse: n groups of FP64 values from the pinned slot.
template <int S>
__global__ __launch_bounds__(THREADS) void k_write_linear(void* mom, Linear L, int k0, uint32_t j0, uint32_t n,
                                                          const f64x4* __restrict__ in) {
    using W = Word<S>;
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if (i >= n) return;
    int k = k0;
    uint32_t j = j0;
    plane_group(L, i, k, j);
    const f64x4 v = in[i];
    const float s = L.scale[k];
    const typename W::V w = {W::enc(v.x, s), W::enc(v.y, s), W::enc(v.z, s), W::enc(v.w, s)};
    *(typename W::V*)((typename W::T*)mom + L.node(j) + (size_t)k * L.T) = w;
}

template <int S>
__device__ __forceinline__ void put_node(void* mom, const Linear& L, size_t e, const double m[10]) {
    using W = Word<S>;
    const auto p = (typename W::T*)mom + e;
#pragma unroll
    for (int k = 0; k < 10; k++) p[(size_t)k * L.T] = W::enc(m[k], L.scale[k]);
}

// Stored moments of `n` nodes from density and velocity in the pinned slot
// (four arrays of `pitch` values), one node per thread; FP64, the host's
// expressions.
template <int S>
__global__ __launch_bounds__(THREADS) void k_write_fields(void* mom, Linear L, int q, int mode, double rho0,
                                                          uint32_t j0, uint32_t n, uint32_t pitch,
                                                          const double* __restrict__ in) {
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if (i >= n) return;
    double m[10];
    node_moments(q, mode, rho0, in[i], in[pitch + i], in[2 * pitch + i], in[3 * pitch + i], m);
    put_node<S>(mom, L, L.node(j0 + i / 4) + i % 4, m);
}

// The vortex from per-axis tables of sin k x, cos k x, cos 2 k x (evaluated
// on the host, so the state does not depend on the device's math functions):
// FP64 products in the order of write_taylor_green's host expressions.
struct Vortex {
    const double* tab[3];  // per axis: sin, cos, cos 2 (extent values each)
    int ext[3];
    double amp, u0, rho0;  // amp = 3/16 rho0 u0^2
    __host__ __device__ double rho(int x, int y, int z) const {
        return rho0 + amp * (tab[0][2 * ext[0] + x] + tab[1][2 * ext[1] + y]) * (tab[2][2 * ext[2] + z] + 2.0);
    }
};

template <int S>
__global__ __launch_bounds__(THREADS) void k_write_vortex(void* mom, Linear L, int q, int mode, Vortex v) {
    const uint32_t bx = blockIdx.x % L.ntx, byz = blockIdx.x / L.ntx, by = byz % L.nty, bz = byz / L.nty;
    for (uint32_t t = threadIdx.x; t < L.T; t += THREADS) {
        const int x = (int)((bx << L.lx) + (t & ((1u << L.lx) - 1)));
        const int y = (int)((by << L.ly) + ((t >> L.lx) & ((1u << L.ly) - 1)));
        const int z = (int)((bz << L.lz) + (t >> (L.lx + L.ly)));
        const double sx = v.tab[0][x], cx = v.tab[0][v.ext[0] + x];
        const double sy = v.tab[1][y], cy = v.tab[1][v.ext[1] + y];
        const double cz = v.tab[2][v.ext[2] + z];
        double m[10];
        node_moments(q, mode, v.rho0, v.rho(x, y, z), v.u0 * sx * cy * cz, -v.u0 * cx * sy * cz, 0.0, m);
        put_node<S>(mom, L, (size_t)blockIdx.x * 10 * L.T + t, m);
    }
}

__global__ __launch_bounds__(THREADS) void k_scale(const double* __restrict__ in, double f, uint32_t n,
                                                   double* __restrict__ out) {
    const uint32_t i = blockIdx.x * THREADS + threadIdx.x;
    if (i < n) __builtin_nontemporal_store(in[i] * f, &out[i]);
}

unsigned blocks(uint32_t n) { return (n + THREADS - 1) / THREADS; }

#define MRLBM_BY_STORAGE(KERNEL, GRID, ...)                                                 \
    do {                                                                                    \
        if (c->p.storage == MRLBM_STORE_FP32)                                               \
            hipLaunchKernelGGL(KERNEL<0>, dim3(GRID), dim3(THREADS), 0, c->stream, __VA_ARGS__); \
        else if (c->p.storage == MRLBM_STORE_FP16)                                          \
            hipLaunchKernelGGL(KERNEL<1>, dim3(GRID), dim3(THREADS), 0, c->stream, __VA_ARGS__); \
        else                                                                                \
            hipLaunchKernelGGL(KERNEL<2>, dim3(GRID), dim3(THREADS), 0, c->stream, __VA_ARGS__); \
    } while (0)

// Chunks of at most `per` of `total` units.
struct Chunks {
    uint64_t total, per;
    size_t count() const { return (size_t)((total + per - 1) / per); }
    uint64_t first(size_t k) const { return k * per; }
    uint32_t size(size_t k) const {
        const uint64_t f = first(k);
        return (uint32_t)(total - f < per ? total - f : per);
    }
};

// Lowest node index whose density is not positive (NaN included), or N.
size_t first_bad_density(const double* rho, size_t N) {
    const size_t per = 1u << 17;
    const size_t chunks = (N + per - 1) / per;
    const int W = workers_for(chunks);
    std::atomic<size_t> bad{N};
    run_workers(W, [&](int w) {
        for (size_t k = w; k < chunks; k += W) {
            const size_t end = (k + 1) * per < N ? (k + 1) * per : N;
            bool ok = true;
            for (size_t j = k * per; j < end; j++) ok &= rho[j] > 0;
            if (ok) continue;
            size_t j = k * per;
            while (rho[j] > 0) j++;
            size_t cur = bad.load();
            while (j < cur && !bad.compare_exchange_weak(cur, j)) {
            }
            return;  // this worker's later chunks lie higher
        }
    });
    return bad.load();
}

int bad_density(const mrlbm_ctx* c, size_t j) {
    const size_t nx = c->p.nx, ny = c->p.ny;
    return fail(MRLBM_EINVAL, "non-positive density at (%d,%d,%d)", (int)(j % nx), (int)(j / nx % ny),
                (int)(j / (nx * ny)));
}

}  // namespace

namespace mrlbm {

void count_lattices(int d) { g_slots.count(d); }

namespace {

// The first `planes` stored moments, plane k into out[k]; widen(o, in, n,
// plane) files n FP32 values of one plane.
template <typename Widen>
int read_planes(mrlbm_ctx* c, int planes, double* const* out, Widen&& widen) {
    const Linear L = linear_of(c);
    const Chunks ch{(uint64_t)L.groups * planes, SLOT_BYTES / sizeof(f32x4)};
    return pump<true>(
        c, ch.count(),
        [&](size_t k, char* slot) {
            const uint64_t f = ch.first(k);
            const uint32_t n = ch.size(k);
            MRLBM_BY_STORAGE(k_read_linear, blocks(n), c->d_mom, L, (int)(f / L.groups), (uint32_t)(f % L.groups), n,
                             (f32x4*)slot);
            return hipGetLastError();
        },
        [&](size_t k, const char* slot) {
            const float* in = (const float*)slot;
            uint64_t at = 4 * ch.first(k);
            const uint64_t end = at + 4 * (uint64_t)ch.size(k);
            while (at < end) {  // a chunk of a small lattice spans planes
                const uint64_t plane = at / c->N, stop = (plane + 1) * c->N < end ? (plane + 1) * c->N : end;
                widen(out[plane] + (at - plane * c->N), in, (size_t)(stop - at), (int)plane);
                in += stop - at;
                at = stop;
            }
        });
}

}  // namespace

int read_moments_linear(mrlbm_ctx* c, double* out) {
    double* plane[10];
    for (int k = 0; k < 10; k++) plane[k] = out + (size_t)k * c->N;
    return read_planes(c, 10, plane, [](double* o, const float* in, size_t n, int) {
        for (size_t j = 0; j < n; j++) o[j] = in[j];
    });
}

int read_macroscopic_linear(mrlbm_ctx* c, double rho0, double* const out[4]) {
    return read_planes(c, 4, out, [rho0](double* o, const float* in, size_t n, int plane) {
        if (plane == 0)
            for (size_t j = 0; j < n; j++) o[j] = (double)in[j] + rho0;
        else
            for (size_t j = 0; j < n; j++) o[j] = (double)in[j] / 3.0;
    });
}

int write_moments_linear(mrlbm_ctx* c, const double* in) {
    const Linear L = linear_of(c);
    const Chunks ch{(uint64_t)L.groups * 10, SLOT_BYTES / sizeof(f64x4)};
    return pump<false>(
        c, ch.count(),
        [&](size_t k, char* slot) {
            const uint64_t f = ch.first(k);
            const uint32_t n = ch.size(k);
            MRLBM_BY_STORAGE(k_write_linear, blocks(n), c->d_mom, L, (int)(f / L.groups), (uint32_t)(f % L.groups), n,
                             (const f64x4*)slot);
            return hipGetLastError();
        },
        [&](size_t k, char* slot) { std::memcpy(slot, in + 4 * ch.first(k), sizeof(f64x4) * (size_t)ch.size(k)); });
}

int write_fields_linear(mrlbm_ctx* c, int mode, const double* rho, const double* ux, const double* uy,
                        const double* uz) {
    const size_t bad = first_bad_density(rho, c->N);
    if (bad < c->N) return bad_density(c, bad);
    const Linear L = linear_of(c);
    constexpr uint32_t PITCH = SLOT_BYTES / (4 * sizeof(double));  // nodes per slot, a multiple of four
    const Chunks ch{c->N, PITCH};
    const double* src[4] = {rho, ux, uy, uz};
    return pump<false>(
        c, ch.count(),
        [&](size_t k, char* slot) {
            const uint32_t n = ch.size(k);
            MRLBM_BY_STORAGE(k_write_fields, blocks(n), c->d_mom, L, c->p.q, mode, c->p.rho0,
                             (uint32_t)(ch.first(k) / 4), n, PITCH, (const double*)slot);
            return hipGetLastError();
        },
        [&](size_t k, char* slot) {
            for (int a = 0; a < 4; a++)
                std::memcpy((double*)slot + (size_t)a * PITCH, src[a] + ch.first(k), sizeof(double) * ch.size(k));
        });
}

int write_taylor_green(mrlbm_ctx* c, double u0, int mode) {
    // cases/taylorGreen/flow_initialization.inc:1-4 with L = N/(2 pi)
    HIPCHK(hipSetDevice(c->p.device));
    const int ext[3] = {c->p.nx, c->p.ny, c->p.nz};
    const size_t n = 3 * ((size_t)ext[0] + ext[1] + ext[2]);
    std::vector<double> tab;
    try {
        tab.resize(n);
    } catch (const std::bad_alloc&) {
        return fail(MRLBM_ENOMEM, "host memory for the vortex tables exhausted");
    }
    Vortex v{};
    size_t off[3], o = 0;
    for (int a = 0; a < 3; a++) {
        const double k = 2.0 * M_PI / ext[a];
        double* t = &tab[off[a] = o];
        for (int j = 0; j < ext[a]; j++) {
            t[j] = std::sin(k * j);
            t[ext[a] + j] = std::cos(k * j);
            t[2 * ext[a] + j] = std::cos(2 * k * j);
        }
        v.ext[a] = ext[a];
        v.tab[a] = t;
        o += 3 * (size_t)ext[a];
    }
    v.rho0 = c->p.rho0;
    v.u0 = u0;
    v.amp = (3.0 / 16.0) * v.rho0 * u0 * u0;
    // |rho - rho0| <= 6 amp: only a large u0 or a negative rho0 needs the
    // node-by-node check
    if (!(v.rho0 > 0 && 6.0 * v.amp < 0.99 * v.rho0))
        for (int z = 0; z < ext[2]; z++)
            for (int y = 0; y < ext[1]; y++)
                for (int x = 0; x < ext[0]; x++)
                    if (!(v.rho(x, y, z) > 0)) return bad_density(c, x + (size_t)ext[0] * (y + (size_t)ext[1] * z));
    double* d = nullptr;
    HIPCHK(hipMallocAsync((void**)&d, sizeof(double) * n, c->stream));
    hipError_t e = hipMemcpyAsync(d, tab.data(), sizeof(double) * n, hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) {
        for (int a = 0; a < 3; a++) v.tab[a] = d + off[a];
        MRLBM_BY_STORAGE(k_write_vortex, c->ntiles, c->d_mom, linear_of(c), c->p.q, mode, v);
        e = hipGetLastError();
    }
    (void)hipFreeAsync(d, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return fail(MRLBM_EHIP, "initial vortex: %s", hipGetErrorString(e));
    return MRLBM_OK;
}

int read_scaled(mrlbm_ctx* c, const double* d_src, size_t n, double factor, double* out) {
    const Chunks ch{n, SLOT_BYTES / sizeof(double)};
    return pump<true>(
        c, ch.count(),
        [&](size_t k, char* slot) {
            hipLaunchKernelGGL(k_scale, dim3(blocks(ch.size(k))), dim3(THREADS), 0, c->stream, d_src + ch.first(k),
                               factor, ch.size(k), (double*)slot);
            return hipGetLastError();
        },
        [&](size_t k, const char* slot) { std::memcpy(out + ch.first(k), slot, sizeof(double) * ch.size(k)); });
}

}  // namespace mrlbm
