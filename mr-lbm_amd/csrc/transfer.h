// Whole fields between the caller's host arrays (x-fastest, FP64) and the
// block layout in HBM (transfer.hip).
#pragma once

#include <stddef.h>
#include <stdio.h>

struct mrlbm_ctx;

namespace mrlbm {

// Workers for a transfer with `left` chunks to go, on `cpus` processors with
// `running` threads on them (this transfer's workers among them, of which
// there are `have`). One core widens 22 GB/s into memory that is in use
// already and 9 GB/s into fresh pages, four 50 GB/s, eight 76 GB/s (PCIe
// delivers 108 GB/s of widened values): more than eight add nothing, and a
// worker is worth its thread (60 us for eight with their end) from about three
// chunks on. Helpers come for free processors only. Where the program's own
// pool still spins after a parallel loop (OpenMP's does for 7 ms), a helper
// waits for a time slice of 3 ms and the call for the last helper, and two of
// the pool's threads may be left on one processor, which holds up the
// program's next loops (28 ms for four of them). A pass of flow statistics
// whose mean flow 16 OpenMP threads then convert, on 16 processors, ms, median
// [90 %]: one copy and a loop over it / eight workers in any case / this rule:
//   0.26 M nodes   1.58 [1.6]      1.3 [4.0]       1.2 [1.3-1.9]
//   0.44 M         2.30 [2.3]      2.0-4.0 [4.1]   1.7 [1.8]
//   0.66 M         3.3 [3.4]       4.0 [5.3]       2.3 [2.5]
//   1.1 M          5.0-7.0 [7.0]   4.2 [6.5]       3.4-5.5 [5.5]
//   2.5 M         14.4 [15]        8.7 [9-31]      8.6 [8.9]
constexpr int MAX_WORKERS = 8;
constexpr size_t CHUNKS_PER_WORKER = 3;
inline int transfer_workers(size_t left, unsigned cpus, unsigned running, int have) {
    const size_t worth = left / CHUNKS_PER_WORKER < MAX_WORKERS ? left / CHUNKS_PER_WORKER : MAX_WORKERS;
    const size_t room = (size_t)have + (cpus > running ? cpus - running : 0);
    const size_t w = worth < room ? worth : room;
    return w > (size_t)have ? (int)w : have;
}

// Threads that run at this moment, on all processors: the fourth field of
// /proc/loadavg (5 us); ~0u where it cannot be read. On a machine shared with
// other programs theirs count too, which only keeps helpers away.
inline unsigned running_threads() {
    unsigned r = ~0u;
    FILE* const f = fopen("/proc/loadavg", "re");
    if (!f) return r;
    if (fscanf(f, "%*s %*s %*s %u/", &r) != 1) r = ~0u;
    fclose(f);
    return r;
}

// Lattices that live (+1, -1): the process's pinned transfer slots are kept
// while there are any.
void count_lattices(int d);

// Stored moments decoded into out[k * N + x + NX (y + NY z)].
int read_moments_linear(mrlbm_ctx* c, double* out);
// rho0 + (rho - RHO_0), ux, uy, uz: four such planes, each by itself.
int read_macroscopic_linear(mrlbm_ctx* c, double rho0, double* const out[4]);
// Stored moments from the same layout.
int write_moments_linear(mrlbm_ctx* c, const double* in);
// Stored moments from density and velocity fields; refuses a non-positive
// density before anything is written.
int write_fields_linear(mrlbm_ctx* c, int mode, const double* rho, const double* ux, const double* uy,
                        const double* uz);
// Stored moments of the Taylor-Green vortex.
int write_taylor_green(mrlbm_ctx* c, double u0, int mode);
// n FP64 values at d_src (device), each times `factor`.
int read_scaled(mrlbm_ctx* c, const double* d_src, size_t n, double factor, double* out);

}  // namespace mrlbm
