// Stored moments of an initial state, in FP64; one function for the host (the
// uniform state) and the device (whole fields), so that both give the same
// bits (the library is compiled without floating-point contraction).
#pragma once

#include "../../include/mrlbm.h"
#include "lattice.h"

namespace mrlbm {

// Stored (scaled) moments of one node from unscaled macroscopic fields.
__host__ __device__ inline void node_moments(int q, int mode, double rho0, double rho, double ux, double uy, double uz,
                                             double m[10]) {
    double pxx, pxy, pxz, pyy, pyz, pzz;
    if (mode == MRLBM_INIT_EQUILIBRIUM) {
        pxx = ux * ux;
        pxy = ux * uy;
        pxz = ux * uz;
        pyy = uy * uy;
        pyz = uy * uz;
        pzz = uz * uz;
    } else {
        // f_eq(w_i RHO_0, u), summed over the D3Q19 index subsets and divided
        // by rho, as src/lbmInitialization.cu:102-130 does for either lattice.
        double f[19];
        const double uu = ux * ux + uy * uy + uz * uz;
#pragma unroll
        for (int i = 0; i < 19; i++) {
            const int cls = wclass(i);
            const double w = q == 19 ? (cls == 0 ? 1.0 / 3 : (cls == 1 ? 1.0 / 18 : 1.0 / 36))
                                     : (cls == 0 ? 8.0 / 27 : (cls == 1 ? 2.0 / 27 : 1.0 / 54));
            const double uc3 = 3.0 * (ux * cxv(i) + uy * cyv(i) + uz * czv(i));
            f[i] = (w * rho0) * ((1.0 - 1.5 * uu) + uc3 * (1.0 + uc3 * 0.5));
        }
        const double ir = 1.0 / rho, cs2 = 1.0 / 3.0;
        pxx = (f[1] + f[2] + f[7] + f[8] + f[9] + f[10] + f[13] + f[14] + f[15] + f[16]) * ir - cs2;
        pxy = ((f[7] + f[8]) - (f[13] + f[14])) * ir;
        pxz = ((f[9] + f[10]) - (f[15] + f[16])) * ir;
        pyy = (f[3] + f[4] + f[7] + f[8] + f[11] + f[12] + f[13] + f[14] + f[17] + f[18]) * ir - cs2;
        pyz = ((f[11] + f[12]) - (f[17] + f[18])) * ir;
        pzz = (f[5] + f[6] + f[9] + f[10] + f[11] + f[12] + f[15] + f[16] + f[17] + f[18]) * ir - cs2;
    }
    m[0] = rho - rho0;
    m[1] = 3.0 * ux;
    m[2] = 3.0 * uy;
    m[3] = 3.0 * uz;
    m[4] = 4.5 * pxx;
    m[5] = 9.0 * pxy;
    m[6] = 9.0 * pxz;
    m[7] = 4.5 * pyy;
    m[8] = 9.0 * pyz;
    m[9] = 4.5 * pzz;
}

}  // namespace mrlbm
