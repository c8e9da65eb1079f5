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
// 0.95 s for the moments of 256^3 FP32 (1.34 GB as FP64; now 22 ms) and
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

// Runs step() until it returns false, on the caller's thread and on helpers
// that join it as processors are free for them: transfer_workers says how
// many, asked after the caller's second step and after every eighth from there
// on (left() is the number of chunks to go). Before a helper starts, grow()
// provides for it on the caller's thread; the helper calls enter() first.
// Either may decline.
template <typename Left, typename Grow, typename Enter, typename Step>
void run_workers(Left&& left, Grow&& grow, Enter&& enter, Step&& step) {
    std::thread th[MAX_WORKERS - 1];
    int have = 1;
    auto helper = [&] {
        if (enter())
            while (step()) {
            }
    };
    auto join_in = [&] {
        const size_t l = left();
        if (l < (have + 1) * CHUNKS_PER_WORKER) return true;
        const int want = transfer_workers(l, std::thread::hardware_concurrency(), running_threads(), have);
        for (; have < want; have++) {
            if (!grow()) return false;
            try {
                th[have - 1] = std::thread(helper);
            } catch (const std::system_error&) {
                return false;
            } catch (const std::bad_alloc&) {
                return false;
            }
        }
        return true;
    };
    bool more = true;
    for (size_t n = 1; step(); n++)
        if (more && n % 8 == 2) more = join_in();
    for (int w = 1; w < have; w++) th[w - 1].join();
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
    hipError_t add() {
        hipError_t e = g_slots.take(&mem[n]);
        if (e != hipSuccess) return e;
        if ((e = hipEventCreateWithFlags(&ev[n], hipEventDisableTiming)) != hipSuccess) {
            g_slots.give(mem[n]);
            return e;
        }
        n++;
        return hipSuccess;
    }
    ~Slots() {
        for (int k = 0; k < n; k++) {
            (void)hipEventDestroy(ev[k]);
            g_slots.give(mem[k]);
        }
    }
};

// Moves `chunks` chunks through pinned slots. DOWN: launch(c, slot) makes the
// device fill the slot, take(c, slot) empties it on the host; otherwise take
// fills it and launch makes the device read it. A worker takes the next chunk
// when it is free, so one that the scheduler holds up keeps back a single
// chunk. Returns when every chunk has arrived and the stream is idle.
template <bool DOWN, typename Launch, typename Take>
int pump(mrlbm_ctx* c, size_t chunks, Launch&& launch, Take&& take) {
    HIPCHK(hipSetDevice(c->p.device));
    if (chunks == 0) return MRLBM_OK;
    Slots slots;
    std::mutex mu;                           // guards what follows
    int spare[2 * MAX_WORKERS], spares = 0;  // slots not in use
    struct Sent {
        int slot;
        size_t chunk;
    } sent[2 * MAX_WORKERS];  // slots the device works on, oldest first
    int head = 0, sents = 0;
    size_t next = 0;  // first chunk not begun
    hipError_t err = hipSuccess;
    // two more slots, for one more worker; one does for the caller
    auto grow = [&] {
        hipError_t e = hipSuccess;
        for (int k = 0; k < 2 && slots.n < 2 * MAX_WORKERS && (size_t)slots.n < chunks; k++) {
            if ((e = slots.add()) != hipSuccess) {
                (void)hipGetLastError();
                break;
            }
            std::lock_guard<std::mutex> lock(mu);
            spare[spares++] = slots.n - 1;
        }
        return e;
    };
    hipError_t e = grow();
    if (slots.n == 0) return fail(MRLBM_ENOMEM, "pinned staging memory: %s", hipGetErrorString(e));
    auto step = [&] {
        std::unique_lock<std::mutex> lock(mu);
        // begin a chunk if a slot is there for it, which is one not in use or,
        // upwards, the one that the device is done with first; otherwise,
        // downwards, finish the oldest
        const bool begin = next < chunks && (spares || (!DOWN && sents));
        const bool wait = begin ? !spares : DOWN && sents;
        if (err != hipSuccess || !(begin || wait)) return false;
        Sent s{};
        if (wait) {
            s = sent[head];
            head = (head + 1) % (2 * MAX_WORKERS);
            sents--;
        } else {
            s.slot = spare[--spares];
        }
        if (begin) s.chunk = next++;
        lock.unlock();
        hipError_t r = wait ? hipEventSynchronize(slots.ev[s.slot]) : hipSuccess;
        if (r == hipSuccess && begin != DOWN) take(s.chunk, slots.mem[s.slot]);
        if (r == hipSuccess && begin) {
            r = launch(s.chunk, slots.mem[s.slot]);
            if (r == hipSuccess) r = hipEventRecord(slots.ev[s.slot], c->stream);
        }
        lock.lock();
        if (r != hipSuccess) err = r;
        if (begin)
            sent[(head + sents++) % (2 * MAX_WORKERS)] = s;
        else
            spare[spares++] = s.slot;
        return true;
    };
    run_workers(
        [&] {
            std::lock_guard<std::mutex> lock(mu);
            return chunks - next;
        },
        [&] { return grow() == hipSuccess; }, [&] { return hipSetDevice(c->p.device) == hipSuccess; }, step);
    // the slots are released below: nothing may still use them
    e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = err;
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
    std::atomic<size_t> bad{N}, next{0};
    auto yes = [] { return true; };
    run_workers([&] { return next < chunks ? chunks - next : 0; }, yes, yes, [&] {
        const size_t k = next++;
        // ranges are begun in ascending order: behind one with a bad node
        // there is nothing to find
        if (k >= chunks || bad < k * per) return false;
        const size_t end = (k + 1) * per < N ? (k + 1) * per : N;
        bool ok = true;
        for (size_t j = k * per; j < end; j++) ok &= rho[j] > 0;
        if (ok) return true;
        size_t j = k * per;
        while (rho[j] > 0) j++;
        size_t cur = bad.load();
        while (j < cur && !bad.compare_exchange_weak(cur, j)) {
        }
        return false;
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
    // also after a failure: the copy may still read the tables
    const hipError_t idle = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = idle;
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
