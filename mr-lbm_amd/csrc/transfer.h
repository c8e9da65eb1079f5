// Whole fields between the caller's host arrays (x-fastest, FP64) and the
// block layout in HBM (transfer.hip).
#pragma once

#include <stddef.h>

struct mrlbm_ctx;

namespace mrlbm {

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
