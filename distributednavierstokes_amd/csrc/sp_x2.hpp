// The spectral x pass by wavefronts for half lengths N = n/2 = N1·N2 with
// N2 <= N1 <= 16: every (y, z) line is transformed by N1 lanes of one
// wavefront (64 / N1 lines at a time), its points in registers.
#pragma once

#include "common.hpp"

namespace dns {

// mode 0: c2r of P[.., 0:3], the velocity bound, the six products (plus the
//         physical stress tau when given), r2c of each into P[.., 0:6];
//      1: c2r of P[.., 0:3] into phys;  2: r2c of phys into P[.., 0:3];
//      3: c2r and the velocity bound only
// (XMID_RHS, XMID_C2R, XMID_R2C, XMID_VMAX of spectral_kernels.hpp).
template <typename T> struct X2Args {
    cplx<T> *P;
    T *phys;         // (n, n, n, 3)
    const T *tau;    // (n, n, n, 6) added to the products, or null
    double *vpart;   // one partial of max Σ_c |v_c| per block, or null
    const cplx<T> *tw, *twx; // exp(-2πi t/N), t < N; exp(-2πi t/n), t <= N
    int n, K, mode;
    int nlines;      // lines of P (n² of phys and tau, which only whole grids pass)
};

}  // namespace dns
