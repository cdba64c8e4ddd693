// Kernel of sp_x2.hpp, instantiated per type and half length by sp_x2_*.hip.
#pragma once

#include "fft_reg.hpp"
#include "sp_x2.hpp"
#include "sp_x2_shapes.hpp"

namespace dns {

// One (y, z) line per N1 lanes.  A transform of N = N1·N2 points is two
// steps with one exchange through the line's LDS storage: with
// i = s + N1 u and k = t + N2 r,
//   X[k] = Σ_s w_N^(s t) w_N1^(s r) Σ_u w_N2^(u t) x[i],
// so lane s takes the DFT over its N2 registers u, the twiddles w_N^(s t),
// and after the exchange lane t (< N2) the DFT over N1 registers; the
// inverse runs the steps in the other order.  The c2r leaves the values
// j = s + N1 u of the three components in the registers of lane s, where the
// products are formed and their r2c starts; physical values reach LDS or HBM
// only in modes 1 and 2.  The exchange keeps element (q, t) at q P1 + t with
// P1 odd, so that both its rows and its columns spread over the banks.  No
// workgroup barrier after the twiddle staging.
//
// What bounds it: the block-wide engine of k_sp_xmid spends three passes of
// two workgroup barriers per transform at 28-84 % of the lanes (n = 384 FP32
// 1.18 ms per launch against 0.28 ms for its bytes at the copy rate); this
// form is bound by VALU issue and HBM together (whole steps of both forms
// stand at the dispatch, SpecImpl::create).
template <typename T, int N1, int N2>
__global__ void __launch_bounds__(256, 2) k_sp_x2(X2Args<T> a)
{
    constexpr int N = N1 * N2, P1 = N2 | 1, LPW = 64 / N1, LS = N1 * P1;
    static_assert(N2 <= N1 && N1 <= 16, "k_sp_x2: N2 <= N1 <= 16");
    extern __shared__ unsigned char smem_raw[];
    cplx<T> *tw2 = reinterpret_cast<cplx<T> *>(smem_raw); // w_N^(q t) at q P1 + t
    cplx<T> *twx = tw2 + LS;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwv = blockDim.x >> 6;
    const int lane = threadIdx.x & 63, lg = lane / N1, t = lane - lg * N1;
    cplx<T> *ex = twx + N + (wv * LPW + (lg < LPW ? lg : 0)) * LS;
    for (int e = threadIdx.x; e < N1 * N2; e += blockDim.x) {
        const int q = e / N2, tt = e - q * N2;
        tw2[q * P1 + tt] = a.tw[q * tt];
    }
    for (int e = threadIdx.x; e < N; e += blockDim.x) twx[e] = a.twx[e];
    __syncthreads();

    const int n = a.n, K = a.K, nlines = a.nlines, sz = (int)sizeof(cplx<T>);
    const int L0 = __builtin_amdgcn_readfirstlane((xcd_block(blockIdx.x, gridDim.x) * nwv + wv) * LPW);
    const int nl = __builtin_amdgcn_readfirstlane(max(0, min(LPW, nlines - L0))); // lines of this wavefront
    const bool mine = lg < nl;
    const bool act = mine && t < N2; // holds N1 points of a line between the steps
    const size_t pstride = (size_t)K * nlines, vstride = (size_t)n * nlines;
    const size_t row0 = (size_t)(nl > 0 ? L0 : 0);
    const uint32_t rowbytes = (uint32_t)nl * K * sz, vbytes = (uint32_t)nl * n * (uint32_t)sizeof(T);
    constexpr int OOB = (int)0x80000000u; // beyond every buffer: reads zero, writes dropped
    const int krow = lg * K;
    const int vrow = mine ? (lg * n + 2 * t) * (int)sizeof(T) : OOB;

    cplx<T> v[3][N2];
    if (a.mode != 2) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bufres row = make_bufres(a.P + row0 * K + c * pstride, rowbytes);
            if (act) {
                cplx<T> z[N1], zn[N1];
#pragma unroll
                for (int r = 0; r < N1; ++r) {
                    const int k = t + N2 * r;
                    z[r] = bload<cplx<T>>(row, k < K ? (krow + k) * sz : OOB, 0);
                    zn[r] = bload<cplx<T>>(row, N - k < K ? (krow + N - k) * sz : OOB, 0);
                }
#pragma unroll
                for (int r = 0; r < N1; ++r) {
                    cplx<T> Xk = z[r], Xn = zn[r];
                    if (r == 0 && t == 0) {
                        Xk.y = T(0);
                        Xn.y = T(0);
                    }
                    const cplx<T> Xc = cconj<T>(Xn);
                    const cplx<T> ev = cadd<T>(Xk, Xc);
                    const cplx<T> od = cmulc<T>(csub<T>(Xk, Xc), twx[t + N2 * r]);
                    z[r] = mk<T>(ev.x - od.y, ev.y + od.x);
                }
                Dft<T, N1, true>::run(z);
                ex[t] = z[0];
#pragma unroll
                for (int q = 1; q < N1; ++q) ex[q * P1 + t] = cmulc<T>(z[q], tw2[q * P1 + t]);
            }
            wave_lds_sync();
#pragma unroll
            for (int u = 0; u < N2; ++u) v[c][u] = ex[t * P1 + u];
            wave_lds_sync();
            Dft<T, N2, true>::run(v[c]);
        }
        if (a.vpart) {
            __shared__ double red[4];
            double mx = 0;
#pragma unroll
            for (int u = 0; u < N2; ++u) {
                mx = fmax(mx, fabs((double)v[0][u].x) + fabs((double)v[1][u].x) + fabs((double)v[2][u].x));
                mx = fmax(mx, fabs((double)v[0][u].y) + fabs((double)v[1][u].y) + fabs((double)v[2][u].y));
            }
            if (!mine) mx = 0;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
            if (lane == 0) red[wv] = mx;
            __syncthreads();
            if (threadIdx.x == 0) {
                for (int w = 1; w < nwv; ++w) mx = fmax(mx, red[w]);
                a.vpart[blockIdx.x] = mx;
            }
        }
        if (a.mode == 3) return;
        if (a.mode == 1) {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const bufres out = make_bufres(a.phys + row0 * n + c * vstride, vbytes);
#pragma unroll
                for (int u = 0; u < N2; ++u) bstore(out, vrow, u * 2 * N1 * (int)sizeof(T), v[c][u]);
            }
            return;
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const bufres in = make_bufres(a.phys + row0 * n + c * vstride, vbytes);
#pragma unroll
            for (int u = 0; u < N2; ++u) v[c][u] = bload<cplx<T>>(in, vrow, u * 2 * N1 * (int)sizeof(T));
        }
    }
#pragma unroll
    for (int p = 0; p < 6; ++p) {
        if (p >= 3 && a.mode == 2) break;
        const int ca = p < 3 ? p : (p == 3 ? 0 : p == 4 ? 1 : 2);
        const int cb = p < 3 ? p : (p == 3 ? 1 : p == 4 ? 2 : 0);
        cplx<T> y[N2];
        if (a.tau) {
            const bufres st = make_bufres(a.tau + row0 * n + p * vstride, vbytes);
#pragma unroll
            for (int u = 0; u < N2; ++u) y[u] = bload<cplx<T>>(st, vrow, u * 2 * N1 * (int)sizeof(T));
#pragma unroll
            for (int u = 0; u < N2; ++u)
                y[u] = mk<T>(v[ca][u].x * v[cb][u].x + y[u].x, v[ca][u].y * v[cb][u].y + y[u].y);
        } else {
#pragma unroll
            for (int u = 0; u < N2; ++u)
                y[u] = p < 3 && a.mode == 2 ? v[p][u] : mk<T>(v[ca][u].x * v[cb][u].x, v[ca][u].y * v[cb][u].y);
        }
        Dft<T, N2, false>::run(y);
        if (mine) {
            ex[t * P1] = y[0];
#pragma unroll
            for (int q = 1; q < N2; ++q) ex[t * P1 + q] = cmul<T>(y[q], tw2[t * P1 + q]);
        }
        wave_lds_sync();
        cplx<T> z[N1];
        if (act) {
#pragma unroll
            for (int q = 0; q < N1; ++q) z[q] = ex[q * P1 + t];
        }
        wave_lds_sync();
        if (act) {
            Dft<T, N1, false>::run(z);
#pragma unroll
            for (int r = 0; r < N1; ++r) ex[t + N2 * r] = z[r];
        }
        wave_lds_sync();
        if (act) {
            const bufres out = make_bufres(a.P + row0 * K + p * pstride, rowbytes);
#pragma unroll
            for (int r = 0; r < N1; ++r) {
                if (N2 * r >= K) break;
                const int k = t + N2 * r;
                const cplx<T> Zk = z[r];
                const cplx<T> Zc = cconj<T>(ex[r == 0 && t == 0 ? 0 : N - k]);
                const cplx<T> sm = cadd<T>(Zk, Zc), df = csub<T>(Zk, Zc);
                const cplx<T> wd = cmul<T>(twx[k], df);
                bstore(out, k < K ? (krow + k) * sz : OOB, 0, mk<T>(T(0.5) * (sm.x + wd.y), T(0.5) * (sm.y - wd.x)));
            }
        }
        wave_lds_sync();
    }
}

template <typename T, int N1, int N2> inline bool sp_x2_go(const X2Args<T> &a, int blocks, int waves, hipStream_t st)
{
    if constexpr (sp_x2_shape<T>(N2)) {
        constexpr int LS = N1 * (N2 | 1), LPW = 64 / N1;
        const size_t lds = sizeof(cplx<T>) * (size_t)(LS + N1 * N2 + waves * LPW * LS);
        hipLaunchKernelGGL((k_sp_x2<T, N1, N2>), dim3(blocks), dim3(64 * waves), lds, st, a);
        return true;
    }
    return false;
}

}  // namespace dns
