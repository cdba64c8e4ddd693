// Pencil passes (line transforms along y or z of arrays whose fastest index
// is kx) by two-step register transforms: n = N1·N2, N2 <= N1 <= 32.
#pragma once

#include "common.hpp"

namespace dns {

enum P2Kind {
    P2_BACK,  // spectral: compact lines (m retained points) -> n points, inverse
    P2_FWD,   // spectral: n points -> retained points, forward, times scale
    P2_STAGE, // spectral: forward y transform of the six products + IF stage
    P2_FULL,  // n points -> n points in place, forward
    P2_FULLI, // the same, inverse
    P2_FOURIER // forward, division by λ1 + λ2 + λ3 (times scale), inverse, in place
};

// Line (kx, y', z') of the grid (tiles of 2^lb consecutive kx, blockIdx.y,
// blockIdx.z) starts at src/dst + kx + by·s1 + bz·s2; its points lie
// `stride` apart.
template <typename T> struct P2Args {
    const cplx<T> *src;
    cplx<T> *dst;
    size_t src1, src2, dst1, dst2;
    int sstride, dstride;
    const cplx<T> *tw; // exp(-2πi t/n), t < n
    int n, K, lb;      // line length, kx extent, log2 of the lines per block
    int kcut, m;       // spectral truncation (P2_BACK, P2_FWD, P2_STAGE)
    T scale;
    // P2_STAGE (fields as StageArgs in spectral_kernels.hpp)
    cplx<T> *uh, *ustart, *du;
    int mode, first; // mode 0: update uh and ustart; 1: write du
    double kfac;
    T a, b, nudcdt, dt;
    // P2_FOURIER
    const double *lam1, *lam2, *lam3;
    double dscale;
};

// Line lengths N1·N2 of P2_STAGE.  Three accumulators per retained output and
// the transform's points fill the registers of longer lines at one wavefront
// per SIMD; a first radix up to 16 holds on longest.  Elsewhere the block
// kernel k_sp_ystage serves (µs per launch of this kernel / of that one, forced
// box on MI355X: FP64 180 90 / 120, 192 120 / 126, 240 213 / 252, 256 229 / 253,
// but 200 193 / 135, 216 247 / 205, 250 345 / 264; FP32 180 32 / 56, 192 51-56 /
// 55, 240 96 / 130, 256 125 / 130, but 200 90 / 66, 250 152 / 137, 288 251 / 207,
// 320 287 / 263, 360 412 / 397, and 324, 384 and 400 equal).
constexpr bool p2_stage_shape(int n1, int n2) { return n1 * n2 <= 180 || (n1 <= 16 && n1 * n2 <= 256); }

// False when no kernel serves (T, n, kind): the caller takes the LDS tiles.
bool p2_launch(P2Kind kind, const P2Args<float> &a, dim3 grid, hipStream_t st);
bool p2_launch(P2Kind kind, const P2Args<double> &a, dim3 grid, hipStream_t st);
// Whether a line length is served for this kind.
template <typename T> bool p2_serves(P2Kind kind, int n);

}  // namespace dns
