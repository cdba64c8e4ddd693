// Small DFTs in registers for the two-step line transforms: radices that are
// products of the primitive ones of fft_lds.hpp (6, 9, 10, 12, 15, 16, 18, 20,
// 24, 25, 27, 32), with their inner twiddles folded to
// constants.
#pragma once

#include "fft_lds.hpp"

namespace dns {

// cos and sin of 2π k / R, reduced to the first octant by integer symmetry
// (multiples of a quarter turn are exact) and summed as Taylor series.
struct TwConst {
    double c, s;
};
constexpr TwConst tw_const(int k, int R)
{
    int num = 8 * (k % R); // the angle is 2π num / (8 R)
    bool sneg = false, cneg = false, swap = false;
    if (num > 4 * R) {
        num = 8 * R - num;
        sneg = true;
    }
    if (num > 2 * R) {
        num = 4 * R - num;
        cneg = true;
    }
    if (num > R) {
        num = 2 * R - num;
        swap = true;
    }
    const long double x = 6.283185307179586476925286766559005768L * (long double)num / (long double)(8 * R);
    long double c = 1, s = x, tc = 1, ts = x;
    for (int i = 1; i < 14; ++i) {
        tc = -tc * x * x / (long double)((2 * i - 1) * (2 * i));
        ts = -ts * x * x / (long double)((2 * i) * (2 * i + 1));
        c += tc;
        s += ts;
    }
    const double cc = (double)(swap ? s : c), ss = (double)(swap ? c : s);
    return TwConst{cneg ? -cc : cc, sneg ? -ss : ss};
}

// z · exp(∓2πi k / R) with the quarter turns as swaps.
template <typename T, int K, int R, bool INV> __device__ __forceinline__ cplx<T> cmul_tw(cplx<T> z)
{
    constexpr TwConst w = tw_const(K, R);
    if constexpr (K % R == 0) return z;
    else if constexpr (4 * K % R == 0 && (4 * K / R) % 4 == 1) return rot_i<T, INV>(z);
    else if constexpr (4 * K % R == 0 && (4 * K / R) % 4 == 2) return mk<T>(-z.x, -z.y);
    else if constexpr (4 * K % R == 0 && (4 * K / R) % 4 == 3) return rot_i<T, !INV>(z);
    else {
        const T c = T(w.c), s = INV ? T(w.s) : T(-w.s);
        return mk<T>(c * z.x - s * z.y, c * z.y + s * z.x);
    }
}

// R = R1·R2 points: DFTs of R1 points over the stride R2, the inner
// twiddles, DFTs of R2 points; output c + R1 d.
template <typename T, int R1, int R2, bool INV> struct DftC {
    template <int A, int C> __device__ static __forceinline__ void column(cplx<T> *v, cplx<T> (&y)[R1][R2])
    {
        if constexpr (C < R1) {
            y[C][A] = cmul_tw<T, A * C, R1 * R2, INV>(y[C][A]);
            column<A, C + 1>(v, y);
        }
    }
    template <int A> __device__ static __forceinline__ void columns(cplx<T> *v, cplx<T> (&y)[R1][R2])
    {
        if constexpr (A < R2) {
            cplx<T> b[R1];
#pragma unroll
            for (int r = 0; r < R1; ++r) b[r] = v[A + R2 * r];
            Dft<T, R1, INV>::run(b);
#pragma unroll
            for (int r = 0; r < R1; ++r) y[r][A] = b[r];
            column<A, 1>(v, y);
            columns<A + 1>(v, y);
        }
    }
    __device__ static __forceinline__ void run(cplx<T> *v)
    {
        cplx<T> y[R1][R2];
        columns<0>(v, y);
#pragma unroll
        for (int c = 0; c < R1; ++c) {
            Dft<T, R2, INV>::run(y[c]);
#pragma unroll
            for (int d = 0; d < R2; ++d) v[c + R1 * d] = y[c][d];
        }
    }
};

template <typename T, bool INV> struct Dft<T, 6, INV> : DftC<T, 2, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 9, INV> : DftC<T, 3, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 10, INV> : DftC<T, 2, 5, INV> {};
template <typename T, bool INV> struct Dft<T, 12, INV> : DftC<T, 4, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 15, INV> : DftC<T, 5, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 16, INV> : DftC<T, 4, 4, INV> {};
template <typename T, bool INV> struct Dft<T, 18, INV> : DftC<T, 6, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 20, INV> : DftC<T, 4, 5, INV> {};
template <typename T, bool INV> struct Dft<T, 24, INV> : DftC<T, 8, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 25, INV> : DftC<T, 5, 5, INV> {};
template <typename T, bool INV> struct Dft<T, 27, INV> : DftC<T, 9, 3, INV> {};
template <typename T, bool INV> struct Dft<T, 32, INV> : DftC<T, 8, 4, INV> {};

}  // namespace dns
