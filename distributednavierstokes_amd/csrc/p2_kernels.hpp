// Kernels of p2.hpp, instantiated per type and line length by p2_*.hip.
//
// A block owns 2^lb consecutive kx lines; thread (b, q) = (tid mod 2^lb,
// tid div 2^lb), q < N1.  With i = j + N2 r and k = s + N1 u,
//   X[k] = Σ_j w_N2^(j u) w_n^(j s) Σ_r w_N1^(r s) x[i]:
// thread (b, j), j < N2, loads its N1 points straight from HBM into
// registers (the lanes of a row read consecutive kx), takes the N1-point
// DFT and the twiddles w_n^(j s), and after one exchange through LDS thread
// (b, s) takes the N2-point DFT and stores its N2 points.  The exchange
// keeps element (s, j) of line b at (s P1 + j) 2^lb + b, P1 odd: the lines of
// a tile are consecutive, so writes and reads touch consecutive banks.
//
// Against the LDS tiles of spectral_kernels.hpp / fv_kernels.hpp this is one
// LDS round trip and two workgroup barriers per transform instead of three
// to five round trips and up to nine barriers, with no index division.
#pragma once

#include "fft_reg.hpp"
#include "p2.hpp"

namespace dns {

template <typename T, int N1, int N2> struct P2 {
    static constexpr int N = N1 * N2, P1 = N2 | 1;
    static constexpr int SZ = (int)sizeof(cplx<T>);
    static constexpr int OOB = (int)0x80000000u; // beyond every buffer: reads zero, writes dropped
    // retained positions lie outside [n/3 + 1, n − n/3 − 1] for every kcut
    // the 2/3 rule admits
    static constexpr bool dead(int lo, int hi) { return lo > N / 3 && hi < N - N / 3; }
    static constexpr bool dead_r(int r) { return dead(N2 * r, N2 * r + N2 - 1); } // first-step register r
    static constexpr bool dead_u(int u) { return dead(N1 * u, N1 * u + N1 - 1); } // second-step register u
    static constexpr int live_u()
    {
        int c = 0;
        for (int u = 0; u < N2; ++u) c += dead_u(u) ? 0 : 1;
        return c;
    }

    // LDS table w_n^(s j) at s N2 + j
    __device__ static void stage(cplx<T> *tw, const cplx<T> *src)
    {
        for (int e = threadIdx.x; e < N; e += blockDim.x) tw[e] = src[(e / N2) * (e % N2)];
    }
    template <bool INV>
    __device__ static __forceinline__ void step1(cplx<T> (&z)[N1], cplx<T> *ex, const cplx<T> *tw, int b, int j, int lb)
    {
        Dft<T, N1, INV>::run(z);
        ex[(j << lb) + b] = z[0];
#pragma unroll
        for (int s = 1; s < N1; ++s) {
            const cplx<T> w = tw[s * N2 + j];
            ex[((s * P1 + j) << lb) + b] = INV ? cmulc<T>(z[s], w) : cmul<T>(z[s], w);
        }
    }
    template <bool INV>
    __device__ static __forceinline__ void step2(cplx<T> (&y)[N2], const cplx<T> *ex, int b, int s, int lb)
    {
#pragma unroll
        for (int j = 0; j < N2; ++j) y[j] = ex[((s * P1 + j) << lb) + b];
        Dft<T, N2, INV>::run(y);
    }
};

template <typename T> __device__ inline uint32_t p2_range(int stride, int count, int nb)
{
    return (uint32_t)(((size_t)stride * (count - 1) + nb) * sizeof(cplx<T>));
}

template <typename T, int N1, int N2> __global__ void __launch_bounds__(16 * N1) k_p2_back(P2Args<T> a)
{
    using F = P2<T, N1, N2>;
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw = reinterpret_cast<cplx<T> *>(smem_raw), *ex = tw + F::N;
    F::stage(tw, a.tw);
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int lb = a.lb, i0 = bx << lb, nb = min(1 << lb, a.K - i0), b = threadIdx.x & ((1 << lb) - 1), q = threadIdx.x >> lb;
    const int shift = (a.n - a.m) * a.sstride * F::SZ;
    const bufres in = make_bufres(a.src + i0 + by * a.src1 + bz * a.src2, p2_range<T>(a.sstride, a.m, nb));
    const bufres out = make_bufres(a.dst + i0 + by * a.dst1 + bz * a.dst2, p2_range<T>(a.dstride, F::N, nb));
    cplx<T> z[N1];
    if (q < N2) {
        const int v0 = (b + a.sstride * q) * F::SZ;
#pragma unroll
        for (int r = 0; r < N1; ++r) {
            if (F::dead_r(r)) {
                z[r] = mk<T>(T(0), T(0));
            } else {
                const int t = q + N2 * r, vs = v0 + N2 * r * a.sstride * F::SZ;
                z[r] = bload<cplx<T>>(in, b >= nb ? F::OOB : t <= a.kcut ? vs : t >= F::N - a.kcut ? vs - shift : F::OOB, 0);
            }
        }
    }
    __syncthreads();
    if (q < N2) F::template step1<true>(z, ex, tw, b, q, lb);
    __syncthreads();
    cplx<T> y[N2];
    F::template step2<true>(y, ex, b, q, lb);
    const int v1 = b < nb ? (b + a.dstride * q) * F::SZ : F::OOB;
#pragma unroll
    for (int u = 0; u < N2; ++u) bstore(out, v1, N1 * u * a.dstride * F::SZ, y[u]);
}

template <typename T, int N1, int N2>
__device__ __forceinline__ void p2_load(cplx<T> (&z)[N1], bufres in, int stride, int q, int b, int nb)
{
    using F = P2<T, N1, N2>;
    const int v0 = b < nb ? (b + stride * q) * F::SZ : F::OOB;
#pragma unroll
    for (int r = 0; r < N1; ++r) z[r] = bload<cplx<T>>(in, v0, N2 * r * stride * F::SZ);
}

template <typename T, int N1, int N2> __global__ void __launch_bounds__(16 * N1) k_p2_fwd(P2Args<T> a)
{
    using F = P2<T, N1, N2>;
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw = reinterpret_cast<cplx<T> *>(smem_raw), *ex = tw + F::N;
    F::stage(tw, a.tw);
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int lb = a.lb, i0 = bx << lb, nb = min(1 << lb, a.K - i0), b = threadIdx.x & ((1 << lb) - 1), q = threadIdx.x >> lb;
    const bufres in = make_bufres(a.src + i0 + by * a.src1 + bz * a.src2, p2_range<T>(a.sstride, F::N, nb));
    const bufres out = make_bufres(a.dst + i0 + by * a.dst1 + bz * a.dst2, p2_range<T>(a.dstride, a.m, nb));
    cplx<T> z[N1];
    if (q < N2) p2_load<T, N1, N2>(z, in, a.sstride, q, b, nb);
    __syncthreads();
    if (q < N2) F::template step1<false>(z, ex, tw, b, q, lb);
    __syncthreads();
    cplx<T> y[N2];
    F::template step2<false>(y, ex, b, q, lb);
    const int v1 = (b + a.dstride * q) * F::SZ, shift = (a.n - a.m) * a.dstride * F::SZ;
#pragma unroll
    for (int u = 0; u < N2; ++u) {
        if (F::dead_u(u)) continue;
        const int k = q + N1 * u, vs = v1 + N1 * u * a.dstride * F::SZ;
        bstore(out, b >= nb ? F::OOB : k <= a.kcut ? vs : k >= F::N - a.kcut ? vs - shift : F::OOB, 0, cscale<T>(y[u], a.scale));
    }
}

template <typename T, int N1, int N2, bool INV> __global__ void __launch_bounds__(16 * N1) k_p2_full(P2Args<T> a)
{
    using F = P2<T, N1, N2>;
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw = reinterpret_cast<cplx<T> *>(smem_raw), *ex = tw + F::N;
    F::stage(tw, a.tw);
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int lb = a.lb, i0 = bx << lb, nb = min(1 << lb, a.K - i0), b = threadIdx.x & ((1 << lb) - 1), q = threadIdx.x >> lb;
    const bufres line = make_bufres(a.dst + i0 + by * a.dst1 + bz * a.dst2, p2_range<T>(a.dstride, F::N, nb));
    cplx<T> z[N1];
    if (q < N2) p2_load<T, N1, N2>(z, line, a.dstride, q, b, nb);
    __syncthreads();
    if (q < N2) F::template step1<INV>(z, ex, tw, b, q, lb);
    __syncthreads();
    cplx<T> y[N2];
    F::template step2<INV>(y, ex, b, q, lb);
    const int v1 = b < nb ? (b + a.dstride * q) * F::SZ : F::OOB;
#pragma unroll
    for (int u = 0; u < N2; ++u) bstore(line, v1, N1 * u * a.dstride * F::SZ, y[u]);
}

// Periodic y solve (src/poisson.jl:43-49, 136-138); lines along y at fixed kz
// = blockIdx.y.  The inverse runs the two steps in the other order, from the
// registers the forward one ends in.
template <typename T, int N1, int N2> __global__ void __launch_bounds__(16 * N1) k_p2_fourier(P2Args<T> a)
{
    using F = P2<T, N1, N2>;
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw = reinterpret_cast<cplx<T> *>(smem_raw), *ex = tw + F::N;
    F::stage(tw, a.tw);
    int bx, by, bz;
    xcd_block3(bx, by, bz);
    const int lb = a.lb, i0 = bx << lb, nb = min(1 << lb, a.K - i0), b = threadIdx.x & ((1 << lb) - 1), q = threadIdx.x >> lb;
    const bufres line = make_bufres(a.dst + i0 + by * a.dst1 + bz * a.dst2, p2_range<T>(a.dstride, F::N, nb));
    cplx<T> z[N1];
    if (q < N2) p2_load<T, N1, N2>(z, line, a.dstride, q, b, nb);
    const double l13 = a.lam1[i0 + min(b, nb - 1)] + a.lam3[by];
    double l2[N2];
#pragma unroll
    for (int u = 0; u < N2; ++u) l2[u] = a.lam2[q + N1 * u];
    __syncthreads();
    if (q < N2) F::template step1<false>(z, ex, tw, b, q, lb);
    __syncthreads();
    cplx<T> y[N2];
    F::template step2<false>(y, ex, b, q, lb);
#pragma unroll
    for (int u = 0; u < N2; ++u) {
        const double lam = l13 + l2[u], f = lam == 0.0 ? 0.0 : a.dscale / lam;
        y[u] = mk<T>(T((double)y[u].x * f), T((double)y[u].y * f));
    }
    // this thread's row of the exchange is its own: no barrier before the writes
    Dft<T, N2, true>::run(y);
#pragma unroll
    for (int t = 0; t < N2; ++t) ex[((q * F::P1 + t) << lb) + b] = t ? cmulc<T>(y[t], tw[q * N2 + t]) : y[t];
    __syncthreads();
    if (q < N2) {
#pragma unroll
        for (int s = 0; s < N1; ++s) z[s] = ex[((s * F::P1 + q) << lb) + b];
        Dft<T, N1, true>::run(z);
        const int v0 = b < nb ? (b + a.dstride * q) * F::SZ : F::OOB;
#pragma unroll
        for (int r = 0; r < N1; ++r) bstore(line, v0, N2 * r * a.dstride * F::SZ, z[r]);
    }
}

// Forward y transform of the six product spectra with the divergence-form
// nonlinear term, the Wray stage and the projection (k_sp_ystage, modes 0 and
// 1; fields as there).  Lines along y at fixed compact kz = blockIdx.y.  Thread
// (b, s) ends every product with its retained outputs k = s + N1 u in
// registers, where du accumulates.
template <typename T, int N1, int N2> __global__ void __launch_bounds__((sizeof(T) == 8 ? 8 : 16) * N1) k_p2_stage(P2Args<T> a)
{
    using F = P2<T, N1, N2>;
    constexpr int LU = F::live_u();
    // the next product's loads overlap this one's second step where the
    // registers hold both beside the accumulators
    constexpr bool PF = (3 * LU + N1 + N2) * (int)(sizeof(cplx<T>) / 4) <= 184;
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw = reinterpret_cast<cplx<T> *>(smem_raw), *ex = tw + F::N;
    F::stage(tw, a.tw);
    int bx, kc;
    xcd_block2(bx, kc);
    const int K = a.K, m = a.m, n = F::N;
    const int lb = a.lb, i0 = bx << lb, nb = min(1 << lb, K - i0), b = threadIdx.x & ((1 << lb) - 1), q = threadIdx.x >> lb;
    const T kx = T(a.kfac * (i0 + b)), kz = T(a.kfac * (kc <= a.kcut ? kc : kc - m));
    auto load = [&](cplx<T>(&z)[N1], int p) {
        const bufres in = make_bufres(a.src + i0 + (size_t)K * n * (kc + (size_t)m * p), p2_range<T>(K, n, nb));
        if (q < N2) p2_load<T, N1, N2>(z, in, K, q, b, nb);
    };
    cplx<T> acc[LU][3];
#pragma unroll
    for (int o = 0; o < LU; ++o)
#pragma unroll
        for (int c = 0; c < 3; ++c) acc[o][c] = mk<T>(T(0), T(0));
    cplx<T> z[N1];
    load(z, 0);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        if (q < N2) F::template step1<false>(z, ex, tw, b, q, lb);
        if (PF && p < 5) load(z, p + 1);
        __syncthreads();
        cplx<T> y[N2];
        F::template step2<false>(y, ex, b, q, lb);
        __syncthreads();
        int o = 0;
#pragma unroll
        for (int u = 0; u < N2; ++u) {
            if (F::dead_u(u)) continue;
            const int k = q + N1 * u;
            const cplx<T> sg = cscale<T>(y[u], a.scale);
            const T ky = T(a.kfac * (2 * k < n ? k : k - n));
            // −i k σ  =  (k σ.y, −k σ.x)
            auto add = [&](int c, T kk) { acc[o][c] = cadd<T>(acc[o][c], mk<T>(kk * sg.y, -kk * sg.x)); };
            if (p == 0) add(0, kx);          // σxx
            if (p == 1) add(1, ky);          // σyy
            if (p == 2) add(2, kz);          // σzz
            if (p == 3) add(0, ky), add(1, kx); // σxy
            if (p == 4) add(1, kz), add(2, ky); // σyz
            if (p == 5) add(0, kz), add(2, kx); // σzx
            ++o;
        }
        // (accumulated here, not sunk with the products' values into the epilogue)
#pragma unroll
        for (int i = 0; i < LU; ++i)
#pragma unroll
            for (int c = 0; c < 3; ++c) asm volatile("" : "+v"(acc[i][c].x), "+v"(acc[i][c].y));
        if (!PF && p < 5) load(z, p + 1);
    }
    // (recomputed here, not kept live across the products)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int be = tid & ((1 << lb) - 1), qe = tid >> lb;
    int o = 0;
    const size_t cs = (size_t)K * m * m;
#pragma unroll
    for (int u = 0; u < N2; ++u) {
        if (F::dead_u(u)) continue;
        const int o_ = o++;
        const int k = qe + N1 * u, jc = k <= a.kcut ? k : k - (n - m);
        if (!(be < nb && (k <= a.kcut || k >= n - a.kcut))) continue;
        const size_t base = (size_t)(i0 + be) + (size_t)K * (jc + (size_t)m * kc);
        if (a.mode == 1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) a.du[base + c * cs] = acc[o_][c];
            continue;
        }
        const T ky = T(a.kfac * (k <= a.kcut ? k : k - n));
        const T kk = kx * kx + ky * ky + kz * kz;
        const T phi = exp(-a.nudcdt * kk);
        cplx<T> w[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const cplx<T> s0 = a.first ? a.uh[base + c * cs] : a.ustart[base + c * cs];
            const cplx<T> d = acc[o_][c];
            const T at = a.a * a.dt, bt = a.b * a.dt;
            w[c] = mk<T>(phi * (s0.x + at * d.x), phi * (s0.y + at * d.y));
            a.ustart[base + c * cs] = mk<T>(phi * (s0.x + bt * d.x), phi * (s0.y + bt * d.y));
        }
        // projection û ← û − k (k·û)/|k|², k = 0 untouched
        cplx<T> pr = mk<T>(T(0), T(0));
        if (kk != T(0))
            pr = mk<T>((kx * w[0].x + ky * w[1].x + kz * w[2].x) / kk, (kx * w[0].y + ky * w[1].y + kz * w[2].y) / kk);
        a.uh[base] = mk<T>(w[0].x - kx * pr.x, w[0].y - kx * pr.y);
        a.uh[base + cs] = mk<T>(w[1].x - ky * pr.x, w[1].y - ky * pr.y);
        a.uh[base + 2 * cs] = mk<T>(w[2].x - kz * pr.x, w[2].y - kz * pr.y);
    }
}

template <typename T, int N1, int N2> inline bool p2_go(int kind, const P2Args<T> &a, dim3 grid, hipStream_t st)
{
    using F = P2<T, N1, N2>;
    const dim3 blk(N1 << a.lb);
    const size_t lds = sizeof(cplx<T>) * ((size_t)F::N + ((size_t)(N1 * F::P1) << a.lb));
    switch (kind) {
        case P2_BACK: hipLaunchKernelGGL((k_p2_back<T, N1, N2>), grid, blk, lds, st, a); return true;
        case P2_FWD: hipLaunchKernelGGL((k_p2_fwd<T, N1, N2>), grid, blk, lds, st, a); return true;
        case P2_STAGE:
            if constexpr (p2_stage_shape(N1, N2)) {
                hipLaunchKernelGGL((k_p2_stage<T, N1, N2>), grid, blk, lds, st, a);
                return true;
            }
            return false;
        case P2_FULL: hipLaunchKernelGGL((k_p2_full<T, N1, N2, false>), grid, blk, lds, st, a); return true;
        case P2_FULLI: hipLaunchKernelGGL((k_p2_full<T, N1, N2, true>), grid, blk, lds, st, a); return true;
        case P2_FOURIER: hipLaunchKernelGGL((k_p2_fourier<T, N1, N2>), grid, blk, lds, st, a); return true;
    }
    return false;
}

}  // namespace dns
