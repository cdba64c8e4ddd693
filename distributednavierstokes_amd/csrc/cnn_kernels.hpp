// BF16 MFMA kernels of the sub-filter-stress CNN closure (gfx950): 3×3×3
// periodic convolutions as implicit GEMMs, erf-GELU, MSE loss and Adam.
//
// Activations are channels-last BF16 arrays act[v][c], v = x + M(y + M(z + M b)),
// with the channel count padded to a multiple of 8.  Weights are BF16
// W[o][n][k] (o = 0..26 the offset (dx, dy, dz) = (o%3−1, (o/3)%3−1, o/9−1),
// n = output channel padded to a multiple of 32, k = input channel, contiguous)
// for the forward pass, and the transposed copy WT[o][k][n] for the data
// gradient.  FP32 master weights and Adam moments live beside them.
//
// MFMA: v_mfma_f32_32x32x16_bf16 (wave64): C[32×32] += A[32×16]·B[16×32]; lane l
// supplies A[l%32][8(l/32)..+7] and B[8(l/32)..+7][l%32]; it receives
// C[8(r/4) + 4(l/32) + r%4][l%32] in accumulator r = 0..15.  (The voxel-tile
// kernels k_conv and k_conv_wgrad take v_mfma_f32_32x32x8_bf16: 4 values a lane.)
#pragma once

#include "common.hpp"

namespace dns {

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
// 16-byte register vector for staged loads: a native vector type, so arrays
// of them stay in registers (HIP's uint4 is a struct whose copies are
// memcpys, which keeps such arrays in scratch memory)
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));

__device__ inline unsigned short f2bf(float f)
{
    // round to nearest even
    unsigned int u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)(u >> 16) | ((u & 0xffff) ? 0x40 : 0);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}
__device__ inline float bf2f(unsigned short h) { return __uint_as_float(((unsigned int)h) << 16); }

// Normal CDF Φ(x) = ½(1 + erf(x/√2)) with erf from Abramowitz & Stegun
// 7.1.26 (|error| ≤ 1.5e-7): erf(u) = 1 − t(a1 + t(a2 + t(a3 + t(a4 + t a5))))
// e^{−u²}, t = 1/(1 + p u), u ≥ 0, on the hardware reciprocal and exp2;
// the tail ½ t(…) e^{−u²} is used directly for x < 0 (no cancellation).
// ex returns e^{−x²/2}, which the GELU derivative shares.  The activations
// are rounded to BF16 (2^−8) after every layer, far above this error.
__device__ inline float phi_cdf(float x, float &ex)
{
    const float u = fabsf(x) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, u, 1.0f));
    ex = __expf(-0.5f * x * x);
    const float poly =
        t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 1.061405429f, -1.453152027f), 1.421413741f), -0.284496736f), 0.254829592f);
    const float tail = 0.5f * poly * ex; // ½ erfc(u)
    return x >= 0.0f ? 1.0f - tail : tail;
}
__device__ inline float gelu_f(float x)
{
    float ex;
    return x * phi_cdf(x, ex);
}
__device__ inline float gelu_d(float x)
{
    float ex;
    const float c = phi_cdf(x, ex);
    return c + x * 0.39894228040143268f * ex;
}

struct ConvGeom {
    int M;     // grid points per direction
    int B;     // batch
    long V;    // B M³ voxels
};

// Neighbour voxel of v at offset o (sign = +1: v + d, −1: v − d), periodic.
__device__ inline long conv_nb(long v, int o, int sign, const ConvGeom &g)
{
    const int M = g.M;
    int x = (int)(v % M);
    long r = v / M;
    int y = (int)(r % M);
    r /= M;
    int z = (int)(r % M);
    long b = r / M;
    const int dx = (o % 3 - 1) * sign, dy = ((o / 3) % 3 - 1) * sign, dz = (o / 9 - 1) * sign;
    x += dx;
    y += dy;
    z += dz;
    x = x < 0 ? x + M : (x >= M ? x - M : x);
    y = y < 0 ? y + M : (y >= M ? y - M : y);
    z = z < 0 ? z + M : (z >= M ? z - M : z);
    return x + (long)M * (y + (long)M * (z + (long)M * b));
}

// out[v][n] = Σ_o Σ_k W[o][n][k] · in[v + sign·d_o][k]   (+ epilogue)
//   EPI 0: forward hidden layer: z = acc + bias → zbuf (BF16; null: not kept), a = gelu(z) → out (BF16)
//   EPI 1: forward output layer: y = acc + bias → yout (FP32, nout channels)
//   EPI 2: data gradient: d = acc · gelu'(zprev[v][n]) → out (BF16)
// Block: 4 waves; tile (32·WM voxels) × (32·WN channels), WM·WN = 4.
// KIN = channels of `in` (multiple of 8), NP = padded output channels
// (multiple of 32) = row count of W, NOUT = channels stored.
struct ConvArgs {
    const unsigned short *in;
    const unsigned short *W;
    const float *bias;
    const unsigned short *zprev;
    unsigned short *out;
    unsigned short *zbuf;
    float *yout;
    int kin, np, nout, ldo; // ldo: channel stride of out/zbuf/yout/zprev
    int sign;
};

template <int WM, int WN, int EPI>
__global__ void __launch_bounds__(256) k_conv(ConvArgs a, ConvGeom g)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const long v0 = (long)blockIdx.x * (32 * WM) + 32 * wm;
    const int n0 = blockIdx.y * (32 * WN) + 32 * wn;
    const int row = lane & 31, kh = 4 * (lane >> 5);
    const long v = v0 + row;
    const bool vok = v < g.V;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    if (n0 < a.np) {
        for (int o = 0; o < 27; ++o) {
            const long nb = vok ? conv_nb(v, o, a.sign, g) : 0;
            const unsigned short *ap = a.in + nb * a.kin + kh;
            const unsigned short *bp = a.W + ((size_t)o * a.np + n0 + row) * a.kin + kh;
            for (int k0 = 0; k0 < a.kin; k0 += 8) {
                bf16x4 av, bv;
                if (vok) {
                    const uint2 raw = *reinterpret_cast<const uint2 *>(ap + k0);
                    av = __builtin_bit_cast(bf16x4, raw);
                } else {
                    av = bf16x4{0, 0, 0, 0};
                }
                const uint2 rawb = *reinterpret_cast<const uint2 *>(bp + k0);
                bv = __builtin_bit_cast(bf16x4, rawb);
                acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(av, bv, acc, 0, 0, 0);
            }
        }
    }
    // epilogue: accumulator r holds row 8(r/4) + 4(lane/32) + r%4, column lane%32
    const int col = n0 + (lane & 31);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int rr = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const long vv = v0 + rr;
        if (vv >= g.V || col >= a.nout) continue;
        const float c = acc[r];
        if (EPI == 0) {
            const float z = c + a.bias[col];
            if (a.zbuf) a.zbuf[vv * a.ldo + col] = f2bf(z);
            a.out[vv * a.ldo + col] = f2bf(gelu_f(z));
        } else if (EPI == 1) {
            a.yout[vv * a.ldo + col] = c + a.bias[col];
        } else {
            const float zp = bf2f(a.zprev[vv * a.ldo + col]);
            a.out[vv * a.ldo + col] = f2bf(c * gelu_d(zp));
        }
    }
}

// Same convolution on v_mfma_f32_32x32x16_bf16 (gfx950): each lane feeds 8
// consecutive channels (one 16-byte load per operand), and each wave owns a
// (32·MB voxels) × (32·NB channels) tile so every A load feeds NB MFMAs and
// every B load MB.  Block: 4 waves stacked along the voxels.  KIN must be a
// multiple of 16 and NP a multiple of 32·NB (one block column per 32·NB).
// The k order inside an MFMA is the same permutation for A and B, so the
// products do not depend on how the hardware assigns k to lanes.
template <int MB, int NB, int EPI>
__global__ void __launch_bounds__(256) k_conv16(ConvArgs a, ConvGeom g)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long vbase = ((long)blockIdx.x * 4 + wave) * (32 * MB);
    const int n0 = blockIdx.y * (32 * NB);
    const int row = lane & 31, kh = 8 * (lane >> 5);
    long vrow[MB];
    bool vok[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        vrow[mb] = vbase + 32 * mb + row;
        vok[mb] = vrow[mb] < g.V;
    }
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    const uint4 zero4 = make_uint4(0u, 0u, 0u, 0u);
    for (int o = 0; o < 27; ++o) {
        const unsigned short *ap[MB];
        const unsigned short *bp[NB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
            ap[mb] = a.in + (vok[mb] ? conv_nb(vrow[mb], o, a.sign, g) : 0) * a.kin + kh;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) bp[nb] = a.W + ((size_t)o * a.np + n0 + 32 * nb + row) * a.kin + kh;
        for (int k0 = 0; k0 < a.kin; k0 += 16) {
            bf16x8 av[MB], bv[NB];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                av[mb] = __builtin_bit_cast(bf16x8, vok[mb] ? *reinterpret_cast<const uint4 *>(ap[mb] + k0) : zero4);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) bv[nb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(bp[nb] + k0));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mb], bv[nb], acc[mb][nb], 0, 0, 0);
        }
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int col = n0 + 32 * nb + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const long vv = vbase + 32 * mb + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (vv >= g.V || col >= a.nout) continue;
                const float c = acc[mb][nb][r];
                if (EPI == 0) {
                    const float z = c + a.bias[col];
                    if (a.zbuf) a.zbuf[vv * a.ldo + col] = f2bf(z);
                    a.out[vv * a.ldo + col] = f2bf(gelu_f(z));
                } else if (EPI == 1) {
                    a.yout[vv * a.ldo + col] = c + a.bias[col];
                } else {
                    const float zp = bf2f(a.zprev[vv * a.ldo + col]);
                    a.out[vv * a.ldo + col] = f2bf(c * gelu_d(zp));
                }
            }
        }
}

// Row-staged convolution: a block owns 4 consecutive x-rows (y0..y0+3 at
// fixed z, b) of M = 32·MB voxels, one row per wave; for each of the three
// z offsets it stages the input rows y0−1..y0+4 of plane z + sign·dz in LDS
// (voxel stride kin + 8 halves, so the 16-byte fragment reads of one wave
// spread over the banks), then runs the nine (dx, dy) offsets from LDS with
// the x wrap applied per lane.  Weights stream from L2; each wave keeps a
// (32·MB voxels) × (32·NB channels) accumulator, so every fragment feeds MB
// or NB MFMAs.  Epilogues as k_conv.  Grid (M/4, M, B) blocks of 256 threads;
// LDS 6·M·(kin + 8) halves.  Needs M = 32·MB and kin % 16 == 0.
template <int MB, int NB, int EPI>
__global__ void __launch_bounds__(256) k_conv_rows(ConvArgs a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    unsigned short *sa = reinterpret_cast<unsigned short *>(smem_raw);
    constexpr int M = 32 * MB;
    const int KS = a.kin + 8; // voxel stride in LDS (halves)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 31, h = lane >> 5;
    const int y0 = blockIdx.x * 4, z = blockIdx.y, b = blockIdx.z;
    const int n0 = 0;
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    const int kc8 = a.kin / 8;
    for (int dzi = 0; dzi < 3; ++dzi) {
        const int zs = (z + a.sign * (dzi - 1) + M) % M;
        __syncthreads();
        // stage rows y0-1 .. y0+4 of plane zs
        for (int e = threadIdx.x; e < 6 * M * kc8; e += blockDim.x) {
            const int c8 = e % kc8, t = e / kc8, x = t % M, rr = t / M;
            const int ys = (y0 - 1 + rr + M) % M;
            const long v = x + (long)M * (ys + (long)M * (zs + (long)M * b));
            *reinterpret_cast<uint4 *>(sa + (rr * M + x) * KS + 8 * c8) =
                *reinterpret_cast<const uint4 *>(a.in + v * a.kin + 8 * c8);
        }
        __syncthreads();
        for (int dyi = 0; dyi < 3; ++dyi) {
            const int rr = wave + 1 + a.sign * (dyi - 1); // staged row of this wave's neighbour
            for (int dxi = 0; dxi < 3; ++dxi) {
                const int o = dxi + 3 * dyi + 9 * dzi;
                const int dx = a.sign * (dxi - 1);
                const unsigned short *ap[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const int xs = (32 * mb + row + dx + M) % M;
                    ap[mb] = sa + (rr * M + xs) * KS + 8 * h;
                }
                const unsigned short *bp[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) bp[nb] = a.W + ((size_t)o * a.np + n0 + 32 * nb + row) * a.kin + 8 * h;
                for (int k0 = 0; k0 < a.kin; k0 += 16) {
                    bf16x8 av[MB], bv[NB];
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        bv[nb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(bp[nb] + k0));
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                        av[mb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(ap[mb] + k0));
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[mb], bv[nb], acc[mb][nb], 0, 0, 0);
                }
            }
        }
    }
    const long vrow = (long)M * ((y0 + wave) + (long)M * (z + (long)M * b));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int col = n0 + 32 * nb + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const long vv = vrow + 32 * mb + 8 * (r >> 2) + 4 * h + (r & 3);
                if (col >= a.nout) continue;
                const float c = acc[mb][nb][r];
                if (EPI == 0) {
                    const float zz = c + a.bias[col];
                    if (a.zbuf) a.zbuf[vv * a.ldo + col] = f2bf(zz);
                    a.out[vv * a.ldo + col] = f2bf(gelu_f(zz));
                } else if (EPI == 1) {
                    a.yout[vv * a.ldo + col] = c + a.bias[col];
                } else {
                    const float zp = bf2f(a.zprev[vv * a.ldo + col]);
                    a.out[vv * a.ldo + col] = f2bf(c * gelu_d(zp));
                }
            }
        }
}

// Epilogue of a wavefront's accumulators acc[mb][nb] (the MFMAs take the
// weights as A and the voxels as B, so lane l has voxel vox[mb] and, in
// accumulators 4g..4g+3, the four consecutive channels
// 32·nb + 8g + 4(l / 32) + 0..3, which leave as one 8-byte store per group,
// converted to BF16 in pairs by the hardware (round to nearest even)).
// EPI as k_conv; vox < 0: nothing stored.
template <int MB, int NB, int EPI>
__device__ __forceinline__ void conv_epilogue(const f32x16 (&acc)[MB][NB], const long (&vox)[MB], const ConvArgs &a, int h)
{
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const long vv = vox[mb];
        if (vv < 0) continue;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq) {
                const int c0 = 32 * nb + 8 * gq + 4 * h;
                float v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = acc[mb][nb][4 * gq + k];
                if (EPI == 1) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (c0 + k < a.nout) a.yout[vv * a.ldo + c0 + k] = v[k] + a.bias[c0 + k];
                    continue;
                }
                if (c0 >= a.nout) continue; // nout is a multiple of 4 for the BF16 outputs
                const size_t off = (size_t)vv * a.ldo + c0;
                if (EPI == 0) {
                    float zz[4], gg[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        zz[k] = v[k] + a.bias[c0 + k];
                        gg[k] = gelu_f(zz[k]);
                    }
                    const bf16x4v zb = {(__bf16)zz[0], (__bf16)zz[1], (__bf16)zz[2], (__bf16)zz[3]};
                    const bf16x4v gb = {(__bf16)gg[0], (__bf16)gg[1], (__bf16)gg[2], (__bf16)gg[3]};
                    if (a.zbuf) *reinterpret_cast<bf16x4v *>(a.zbuf + off) = zb;
                    *reinterpret_cast<bf16x4v *>(a.out + off) = gb;
                } else {
                    const bf16x4v zp = *reinterpret_cast<const bf16x4v *>(a.zprev + off);
                    float d[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) d[k] = v[k] * gelu_d((float)zp[k]);
                    const bf16x4v db = {(__bf16)d[0], (__bf16)d[1], (__bf16)d[2], (__bf16)d[3]};
                    *reinterpret_cast<bf16x4v *>(a.out + off) = db;
                }
            }
    }
}

// k_conv_rows with the input channel count KIN (16 or 64) fixed at compile
// time and the next dz plane's input rows loaded into registers while the
// current plane is computed; every wavefront streams its own weight fragments
// from L1/L2 into registers an offset ahead (DNS_CNN_WLDS=0; four times the
// L1 traffic of k_conv_plane, which bound it: forward 5.2 against 3.0 ms per
// 16 × 64³ training step).
template <int MB, int NB, int KIN, int EPI>
__global__ void __launch_bounds__(256) k_conv_rows_pf(ConvArgs a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    unsigned short *sa = reinterpret_cast<unsigned short *>(smem_raw);
    constexpr int M = 32 * MB, KS = KIN + 8, KST = KIN / 16, KC8 = KIN / 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 31, h = lane >> 5;
    const int y0 = blockIdx.x * 4, z = blockIdx.y, b = blockIdx.z;
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    // kernel arguments as locals: the lambdas below capture by reference,
    // and a captured by-value argument struct would be kept in scratch
    const unsigned short *const gin = a.in;
    const int sign = a.sign, np = a.np;
    u32x4 bf[2][NB][KST];
    const unsigned short *wrow = a.W + (size_t)row * KIN + 8 * h;
    auto loadb = [&](int o, u32x4 (&dst)[NB][KST]) __attribute__((always_inline)) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int ks = 0; ks < KST; ++ks)
                dst[nb][ks] = *reinterpret_cast<const u32x4 *>(wrow + ((size_t)o * np + 32 * nb) * KIN + 16 * ks);
    };
    // input rows y0-1 .. y0+4 of plane z + sign·dz: NIT 16-byte pieces per
    // thread, loaded for the next dz while the current one is computed
    constexpr int NPC = 6 * M * KC8, NIT = (NPC + 255) / 256;
    u32x4 st[NIT];
    auto fetch_rows = [&](int dzi) __attribute__((always_inline)) {
        const int zs = (z + sign * (dzi - 1) + M) % M;
#pragma unroll
        for (int i = 0; i < NIT; ++i) {
            const int e = threadIdx.x + 256 * i;
            if (NPC % 256 == 0 || e < NPC) {
                const int c8 = e % KC8, t = e / KC8, x = t % M, rr = t / M;
                const int ys = (y0 - 1 + rr + M) % M;
                const long v = x + (long)M * (ys + (long)M * (zs + (long)M * b));
                st[i] = *reinterpret_cast<const u32x4 *>(gin + v * KIN + 8 * c8);
            }
        }
    };
    loadb(0, bf[0]);
    fetch_rows(0);
#pragma unroll
    for (int dzi = 0; dzi < 3; ++dzi) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NIT; ++i) {
            const int e = threadIdx.x + 256 * i;
            if (NPC % 256 == 0 || e < NPC) {
                const int c8 = e % KC8, t = e / KC8, x = t % M, rr = t / M;
                *reinterpret_cast<u32x4 *>(sa + (rr * M + x) * KS + 8 * c8) = st[i];
            }
        }
        __syncthreads();
        if (dzi < 2) fetch_rows(dzi + 1);
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int o = q + 9 * dzi, cur = o & 1;
            if (o + 1 < 27) loadb(o + 1, bf[cur ^ 1]);
            const int dyi = q / 3, dxi = q % 3;
            const int rr = wave + 1 + a.sign * (dyi - 1);
            const int dx = a.sign * (dxi - 1);
            const unsigned short *ap[MB];
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
                const int xs = (32 * mb + row + dx + M) % M;
                ap[mb] = sa + (rr * M + xs) * KS + 8 * h;
            }
#pragma unroll
            for (int ks = 0; ks < KST; ++ks) {
                bf16x8 av[MB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) av[mb] = *reinterpret_cast<const bf16x8 *>(ap[mb] + 16 * ks);
                bf16x8 wv[NB];
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    wv[nb] = __builtin_bit_cast(bf16x8, bf[cur][nb][ks]);
                }
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[nb], av[mb], acc[mb][nb], 0, 0, 0);
            }
        }
    }
    const long vrow = (long)M * ((y0 + wave) + (long)M * (z + (long)M * b));
    long vox[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) vox[mb] = vrow + 32 * mb + (lane & 31);
    conv_epilogue<MB, NB, EPI>(acc, vox, a, h);
}

// The BF16 epilogues (EPI 0, 2) through LDS: per 32-voxel tile the wavefront
// leaves its FP32 accumulators in its own LDS area [32 voxels][32 NB + 8]
// and takes them back as runs of 8 channels, so that z, a and the previous
// layer's z move as 16 contiguous bytes per lane and whole 128-byte lines per
// eight lanes.  Same arithmetic as conv_epilogue, whose 8-byte stores touch 32
// lines each (16 × 64³: 64 → 64 forward 0.99 → 0.91 ms, 3 → 64 0.58 → 0.45).
// ep: the wavefront's area (conv_ep_floats floats).  zp: the previous
// layer's z of the wavefront's tiles (conv_load_z, EPI 2).
template <int NB> constexpr int conv_ep_floats() { return 32 * (32 * NB + 8); }

// live voxels of a tile (its lanes hold consecutive voxels, live ones first)
__device__ __forceinline__ int conv_live(long vox, int lane) { return __popcll(__ballot(lane < 32 && vox >= 0)); }

template <int MB, int NB>
__device__ __forceinline__ void conv_load_z(bf16x8 (&zp)[MB][2 * NB], const long (&vox)[MB], const ConvArgs &a, int lane)
{
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const long first = __shfl(vox[mb], 0, 64);
        const int live = conv_live(vox[mb], lane);
#pragma unroll
        for (int i = 0; i < 2 * NB; ++i) {
            const int e = lane + 64 * i, v = e / (4 * NB), c0 = 8 * (e % (4 * NB));
            if (v < live && c0 < a.nout) zp[mb][i] = *reinterpret_cast<const bf16x8 *>(a.zprev + (size_t)(first + v) * a.ldo + c0);
        }
    }
}

template <int MB, int NB, int EPI>
__device__ __forceinline__ void conv_epilogue_lds(const f32x16 (&acc)[MB][NB], const long (&vox)[MB], const ConvArgs &a,
                                                  const bf16x8 (&zp)[MB][2 * NB], float *ep, int lane)
{
    constexpr int PITCH = 32 * NB + 8, G8 = 4 * NB; // floats per voxel; 8-channel groups
    const int h = lane >> 5;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        float *row = ep + (lane & 31) * PITCH + 4 * h;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int gq = 0; gq < 4; ++gq)
                *reinterpret_cast<float4 *>(row + 32 * nb + 8 * gq) =
                    make_float4(acc[mb][nb][4 * gq], acc[mb][nb][4 * gq + 1], acc[mb][nb][4 * gq + 2], acc[mb][nb][4 * gq + 3]);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const long first = __shfl(vox[mb], 0, 64);
        const int live = conv_live(vox[mb], lane);
#pragma unroll
        for (int i = 0; i < 32 * G8 / 64; ++i) {
            const int e = lane + 64 * i, v = e / G8, c0 = 8 * (e % G8);
            if (v >= live || c0 >= a.nout) continue;
            const float4 lo = *reinterpret_cast<const float4 *>(ep + v * PITCH + c0);
            const float4 hi = *reinterpret_cast<const float4 *>(ep + v * PITCH + c0 + 4);
            const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            const size_t off = (size_t)(first + v) * a.ldo + c0;
            bf16x8 o, zb;
            if (EPI == 0) {
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const float zz = x[k] + a.bias[c0 + k];
                    zb[k] = (__bf16)zz;
                    o[k] = (__bf16)gelu_f(zz);
                }
                if (a.zbuf) *reinterpret_cast<bf16x8 *>(a.zbuf + off) = zb;
            } else {
#pragma unroll
                for (int k = 0; k < 8; ++k) o[k] = (__bf16)(x[k] * gelu_d((float)zp[mb][i][k]));
            }
            *reinterpret_cast<bf16x8 *>(a.out + off) = o;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Convolution by runs of 256 consecutive voxels v = x + M y of one (z, b)
// plane: each of the four wavefronts takes 64 of them as two 32-voxel tiles
// (parts of a row at M = 64, whole rows at 32, row pairs at 16, and runs
// across row ends at any other M) times 32·NB channels.  The rows the run and
// its y neighbours touch are staged once per dz plane (for a compile-time M
// the next plane's rows are in flight meanwhile).
// Weights: at KIN = 64 each offset's block is loaded an offset ahead into a
// double-buffered LDS copy (one barrier per offset); at KIN = 16 the blocks of
// all 27 offsets (27 NP 32 bytes) are staged once and no barrier separates
// the offsets.  Writing the results as whole lines through LDS
// (conv_epilogue_lds) took the 3 → 64 and 6 → 64 layers of 16 × 64³ from 0.58
// to 0.45 ms, 64 → 64 forward from 0.99 to 0.91.  Both operands are kept
// so that the lanes of a fragment read spread over the banks: rows of
// KIN + 8 halves at KIN = 64, two planes of 8 channels at KIN = 16.
// Products are accumulated in the order dz, dy, dx, k for every voxel.
// MC = M, or 0: M = g.M at run time, rows copied without the lookahead.
// Grid (ceil(M²/256), M, B).  LDS: conv_plane_lds.
inline size_t conv_plane_rows(int M) { return M % 256 == 0 || 256 % M == 0 ? std::max(256 / M, 1) + 2 : (254 + M) / M + 3; }
inline size_t conv_plane_lds(int M, int np, int kin)
{
    const size_t vox = std::min(conv_plane_rows(M), (size_t)M + 2) * M;
    const bool pipe = M == 16 || M == 32 || M == 64;
    const size_t work = kin == 16 ? 32 * vox + (size_t)27 * np * 32
                                  : vox * 2 * (kin + 8) + (pipe ? (size_t)3 * np * 2 * kin : (size_t)2 * np * 2 * (kin + 8));
    return std::max(work, (size_t)4 * 32 * (np + 8) * sizeof(float)); // the epilogue's four areas
}

template <int MC, int NB, int KIN, int EPI>
__global__ void __launch_bounds__(256) k_conv_plane(ConvArgs a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    unsigned short *sa = reinterpret_cast<unsigned short *>(smem_raw);
    constexpr bool WALL = KIN == 16;         // all weights staged once
    constexpr bool PIPE = !WALL && MC != 0;  // fragments one k step ahead, three weight buffers
    constexpr int MB = 2, KST = KIN / 16, KC8 = KIN / 8, NP = 32 * NB, KS = KIN + 8;
    const int M = MC ? MC : g.M, MM = M * M;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = lane & 31, h = lane >> 5;
    const int v0 = blockIdx.x * 256, z = blockIdx.y, b = blockIdx.z;
    const int ylo = v0 / M, yhi = min(v0 + 255, MM - 1) / M, nvox = (yhi - ylo + 3) * M; // staged rows ylo − 1 … yhi + 1
    f32x16 acc[MB][NB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0.0f;
    // kernel arguments as locals: the lambdas below capture by reference,
    // and a captured by-value argument struct would be kept in scratch
    const unsigned short *const gin = a.in, *const gw = a.W;
    const int sign = a.sign;

    // half-word offset of (staged voxel, 8-channel group) in LDS
    auto at = [&](int t, int c8) { return WALL ? (c8 * nvox + t) * 8 : t * KS + 8 * c8; };
    unsigned short *sw = sa + (WALL ? 16 * nvox : KS * nvox);

    // this lane's staged voxel for (tile, dx); dy adds dy·M voxels
    int base[MB][3];
    long vox[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int v = v0 + 64 * wave + 32 * mb + row, vc = min(v, MM - 1), y = vc / M, x = vc - y * M;
        vox[mb] = v < MM ? v + (long)MM * (z + (long)M * b) : -1;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int xs = x + sign * (d - 1), xw = xs < 0 ? xs + M : xs >= M ? xs - M : xs;
            base[mb][d] = at((y - ylo + 1) * M + xw, h);
        }
    }
    const int vstep = M * (WALL ? 8 : KS); // halves per row

    auto piece = [&](int e, int dzi) __attribute__((always_inline)) {
        const int c8 = e % KC8, t = e / KC8, rr = t / M, x = t - rr * M;
        int ys = ylo - 1 + rr, zs = z + sign * (dzi - 1);
        ys = ys < 0 ? ys + M : ys >= M ? ys - M : ys;
        zs = zs < 0 ? zs + M : zs >= M ? zs - M : zs;
        return *reinterpret_cast<const u32x4 *>(gin + ((size_t)x + (size_t)M * (ys + (size_t)M * (zs + (size_t)M * b))) * KIN +
                                                8 * c8);
    };
    constexpr int NPC = MC ? (256 / (MC ? MC : 1) + 2) * MC * KC8 : 0, NIT = MC ? (NPC + 255) / 256 : 1;
    u32x4 st[NIT];
    auto fetch_rows = [&](int dzi) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NIT; ++i) {
            const int e = tid + 256 * i;
            if (NPC % 256 == 0 || e < NPC) st[i] = piece(e, dzi);
        }
    };
    auto place = [&](int e, u32x4 v) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4 *>(sa + at(e / KC8, e % KC8)) = v;
    };

    // weights of offset o: 16-byte pieces e = (n, c8)
    constexpr int NPW = NP * KC8, WPI = (NPW + 255) / 256;
    u32x4 wr[WPI];
    auto loadw = [&](int o) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WPI; ++i) {
            const int e = tid + 256 * i;
            if (NPW % 256 == 0 || e < NPW) wr[i] = *reinterpret_cast<const u32x4 *>(gw + ((size_t)o * NPW + e) * 8);
        }
    };
    auto storew = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WPI; ++i) {
            const int e = tid + 256 * i;
            const int n = e / KC8, c8 = e % KC8;
            if (NPW % 256 == 0 || e < NPW)
                *reinterpret_cast<u32x4 *>(PIPE ? sw + (buf * NP + n) * KIN + 8 * (c8 ^ ((n >> 1) & 7))
                                                : sw + (buf * NP + n) * KS + 8 * c8) = wr[i];
        }
    };
    bf16x8 zp[MB][2 * NB]; // in flight during the last dz plane
    if constexpr (MC != 0) fetch_rows(0);
    if constexpr (WALL) {
        // [offset][8-channel group][n]
        batched_for<8, u32x4>(
            27 * NPW, [&](int e) { return *reinterpret_cast<const u32x4 *>(gw + (size_t)e * 8); },
            [&](int e, u32x4 v) {
                const int c8 = e % KC8, n = (e / KC8) % NP, o = e / (KC8 * NP);
                *reinterpret_cast<u32x4 *>(sw + ((size_t)(o * KC8 + c8) * NP + n) * 8) = v;
            });
    } else {
        loadw(0);
        storew(0);
        loadw(1);
        if (PIPE) {
            storew(1);
            loadw(2);
        }
    }
    // PIPE: fragments of k step t = 4 o + ks; (32 nb + row) rows of 8 pieces,
    // piece 2 ks + h of row n at position (2 ks + h) ^ (n / 2 mod 8)
    bf16x8 fa[2][MB], fw[2][NB];
    const int wsw = KIN * row + 8 * (h ^ ((row >> 1) & 7));
    auto frags = [&](int t) __attribute__((always_inline)) {
        const int o = t / KST, ks = t % KST, q = o % 9;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
            fw[t & 1][nb] = *reinterpret_cast<const bf16x8 *>(sw + ((o % 3) * NP + 32 * nb) * KIN + (wsw ^ (16 * ks)));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
            fa[t & 1][mb] = *reinterpret_cast<const bf16x8 *>(sa + base[mb][q % 3] + sign * (q / 3 - 1) * vstep + 16 * ks);
    };
#pragma unroll
    for (int dzi = 0; dzi < 3; ++dzi) {
        if (WALL && dzi > 0) __syncthreads(); // (else the last offset's barrier)
        if constexpr (MC != 0) {
#pragma unroll
            for (int i = 0; i < NIT; ++i) {
                const int e = tid + 256 * i;
                if (NPC % 256 == 0 || e < NPC) place(e, st[i]);
            }
        } else {
            batched_for<8, u32x4>(nvox * KC8, [&](int e) { return piece(e, dzi); }, place);
        }
        __syncthreads();
        if constexpr (MC != 0)
            if (dzi < 2) fetch_rows(dzi + 1);
        if (EPI == 2 && dzi == 2) conv_load_z<MB, NB>(zp, vox, a, lane);
        if constexpr (PIPE) {
            frags(9 * KST * dzi);
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                const int o = q + 9 * dzi;
                // (this buffer was last read in offset o − 1)
                if (o + 2 < 27) storew((o + 2) % 3);
                if (o + 3 < 27) loadw(o + 3);
#pragma unroll
                for (int ks = 0; ks < KST; ++ks) {
                    const int t = KST * o + ks;
                    if (q < 8 || ks + 1 < KST) frags(t + 1);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[t & 1][nb], fa[t & 1][mb], acc[mb][nb], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                __syncthreads();
            }
            continue;
        }
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int o = q + 9 * dzi, cur = o & 1;
            const int dyi = q / 3, dxi = q % 3;
            const int dy = sign * (dyi - 1) * vstep;
#pragma unroll
            for (int ks = 0; ks < KST; ++ks) {
                bf16x8 av[MB], wv[NB];
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    av[mb] = *reinterpret_cast<const bf16x8 *>(sa + base[mb][dxi] + dy + 16 * ks);
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    wv[nb] = *reinterpret_cast<const bf16x8 *>(
                        WALL ? sw + ((o * KC8 + h) * NP + 32 * nb + row) * 8
                             : sw + (cur * NP + 32 * nb + row) * KS + 16 * ks + 8 * h);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv[nb], av[mb], acc[mb][nb], 0, 0, 0);
            }
            if constexpr (!WALL) {
                // the buffer written here was read in offset o − 1, which every
                // wavefront has finished (the barrier at its end)
                if (o + 1 < 27) storew(cur ^ 1);
                if (o + 2 < 27) loadw(o + 2);
                __syncthreads();
            }
        }
    }
    if constexpr (EPI == 1) {
        conv_epilogue<MB, NB, EPI>(acc, vox, a, h);
    } else {
        if (WALL) __syncthreads(); // every wavefront is done with the rows
        conv_epilogue_lds<MB, NB, EPI>(acc, vox, a, zp, reinterpret_cast<float *>(smem_raw) + wave * conv_ep_floats<NB>(), lane);
    }
}

// Output convolution of the LES stress (64 → nout channels, 3 nout <= 32): the three
// dx taps are columns of one product, P[v][(dx, n)] = Σ_{dz, dy, k}
// W[dx, dy, dz][n][k] in[v + (0, dy, dz)][k], and out[v][n] = b[n] +
// Σ_dx P[v + dx][(dx, n)] is formed from LDS at the end.  So 9 taps of a
// 32-column MFMA do what 27 taps of 6 used columns did, with a third of the
// LDS reads: 26 µs against 36 for one 64³ sample (k_conv_plane); staging the
// rows of each dz (4.5 times the input through L2) is most of what is left.
// A block takes R = min(256 / M, M) whole rows of one (z, b) plane, four
// wavefronts of two 32-voxel tiles; rows ylo − 1 … ylo + R and the weights of
// one dz are staged at a time (MC = M: the next ones in flight meanwhile).
// Grid (ceil(M / R), M); M <= 256.  LDS: conv_out_lds.
constexpr int CO_KS = 72, CO_PITCH = 33, CO_NMAX = 10; // halves per voxel / weight row, floats per voxel of P, most outputs
inline int conv_out_rows(int M) { return std::min(256 / M, M); }
inline size_t conv_out_lds(int M, int nout)
{
    return std::max((size_t)((conv_out_rows(M) + 2) * M + 9 * nout) * 2 * CO_KS, (size_t)256 * CO_PITCH * sizeof(float));
}

// The result: planar (nout, M³), scale · result, in FP32 or FP64 (one sample; a
// pass of its own took 4.7 µs per stage at 64³, five LES steps 3.83 -> 3.70 ms).
struct StressOut {
    float *f;
    double *d;
    double scale;
};

template <int MC> __global__ void __launch_bounds__(256) k_conv_out(ConvArgs a, StressOut so, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    constexpr int MB = 2, KS = CO_KS;
    const int M = MC ? MC : g.M, R = min(256 / M, M);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = lane & 31, h = lane >> 5;
    const int ylo = blockIdx.x * R, nr = min(R, M - ylo), z = blockIdx.y, nout = a.nout, nj = 3 * nout;
    unsigned short *sa = reinterpret_cast<unsigned short *>(smem_raw), *sw = sa + (R + 2) * M * KS;
    f32x16 acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mb][r] = 0.0f;
    int base[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) base[mb] = (min(64 * wave + 32 * mb + row, nr * M - 1) + M) * KS + 8 * h;
    const int wbase = min(row, nj - 1) * KS + 8 * h;

    const unsigned short *const gin = a.in, *const gw = a.W;
    // staged rows in pieces of 8 channels; weights of one dz in pieces e = (dy, dx, n, c8)
    auto piece = [&](int e, int dzi) __attribute__((always_inline)) {
        const int c8 = e & 7, t = e >> 3, rr = t / M, x = t - rr * M;
        int ys = ylo - 1 + rr, zs = z + dzi - 1;
        ys = ys < 0 ? ys + M : ys >= M ? ys - M : ys;
        zs = zs < 0 ? zs + M : zs >= M ? zs - M : zs;
        return *reinterpret_cast<const u32x4 *>(gin + ((size_t)x + (size_t)M * (ys + (size_t)M * zs)) * 64 + 8 * c8);
    };
    auto place = [&](int e, u32x4 v) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4 *>(sa + (e >> 3) * KS + 8 * (e & 7)) = v;
    };
    auto wpiece = [&](int e, int dzi) __attribute__((always_inline)) {
        const int c8 = e & 7, t = e >> 3, q = t / nout, n = t - q * nout; // q = dx + 3 dy
        return *reinterpret_cast<const u32x4 *>(gw + ((size_t)(9 * dzi + q) * a.np + n) * 64 + 8 * c8);
    };
    auto wplace = [&](int e, u32x4 v) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4 *>(sw + (e >> 3) * KS + 8 * (e & 7)) = v;
    };
    const int np = (nr + 2) * M * 8, npw = 9 * nout * 8;
    constexpr int NIT = MC ? ((256 / (MC ? MC : 1) + 2) * MC * 8 + 255) / 256 : 1, WIT = (9 * CO_NMAX * 8 + 255) / 256;
    u32x4 st[NIT], wr[WIT];
    auto fetch = [&](int dzi) __attribute__((always_inline)) {
        if constexpr (MC != 0) {
#pragma unroll
            for (int i = 0; i < NIT; ++i) st[i] = piece(min(tid + 256 * i, np - 1), dzi);
        }
#pragma unroll
        for (int i = 0; i < WIT; ++i)
            if (tid + 256 * i < npw) wr[i] = wpiece(tid + 256 * i, dzi);
    };
    fetch(0);
#pragma unroll
    for (int dzi = 0; dzi < 3; ++dzi) {
        if (dzi > 0) __syncthreads();
        if constexpr (MC != 0) {
#pragma unroll
            for (int i = 0; i < NIT; ++i)
                if (tid + 256 * i < np) place(tid + 256 * i, st[i]);
        } else {
            batched_for<8, u32x4>(np, [&](int e) { return piece(e, dzi); }, place);
        }
#pragma unroll
        for (int i = 0; i < WIT; ++i)
            if (tid + 256 * i < npw) wplace(tid + 256 * i, wr[i]);
        __syncthreads();
        if (dzi < 2) fetch(dzi + 1);
#pragma unroll
        for (int dyi = 0; dyi < 3; ++dyi)
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                const bf16x8 wv = *reinterpret_cast<const bf16x8 *>(sw + dyi * nj * KS + wbase + 16 * ks);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const bf16x8 av = *reinterpret_cast<const bf16x8 *>(sa + base[mb] + (dyi - 1) * M * KS + 16 * ks);
                    acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wv, av, acc[mb], 0, 0, 0);
                }
            }
    }
    __syncthreads();
    float *P = reinterpret_cast<float *>(smem_raw);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = 8 * (r >> 2) + 4 * h + (r & 3);
            if (j < nj) P[(64 * wave + 32 * mb + row) * CO_PITCH + j] = acc[mb][r];
        }
    __syncthreads();
    const size_t v0 = (size_t)M * (ylo + (size_t)M * z);
    const int nv = nr * M;
    const size_t vs = (size_t)M * M * M;
    for (int e = tid; e < nv * nout; e += 256) {
        const int n = e / nv, v = e - n * nv, x = v % M;
        const int vm = x == 0 ? v + M - 1 : v - 1, vp = x == M - 1 ? v - (M - 1) : v + 1;
        const float r = (P[vm * CO_PITCH + n] + P[v * CO_PITCH + nout + n] + P[vp * CO_PITCH + 2 * nout + n]) + a.bias[n];
        if (so.f) so.f[n * vs + v0 + v] = (float)(so.scale * (double)r);
        else so.d[n * vs + v0 + v] = so.scale * (double)r;
    }
}

// Weight gradient of one offset per block-row: for o = blockIdx.y,
// dW[o][n][k] += Σ_{v in chunk} dout[v][n] · in[v + d_o][k], tiles of 64
// voxels staged (transposed) through LDS.  Each block covers a range of
// voxels (blockIdx.x) and the full (NP × KP) output (NP, KP <= 64, multiples
// of 32 after padding), writing FP32 partials part[blockIdx.x][o][n][k].
struct WGradArgs {
    const unsigned short *dout; // [V][ldd]
    const unsigned short *in;   // [V][kin]
    float *part;
    int ldd, nout, kin, np, kp; // np, kp: padded extents of the partial tile
    long chunk;                 // voxels per block
};

__global__ void __launch_bounds__(256) k_conv_wgrad(WGradArgs a, ConvGeom g)
{
    __shared__ unsigned short sd[64][64 + 4]; // [channel n][voxel]
    __shared__ unsigned short si[64][64 + 4]; // [channel k][voxel]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wn = wave & 1, wk = wave >> 1; // 2 × 2 waves of 32 × 32
    const int o = blockIdx.y;
    const long vbeg = (long)blockIdx.x * a.chunk;
    const long vend = min(vbeg + a.chunk, g.V);
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int row = lane & 31, kh = 4 * (lane >> 5);
    for (long vt = vbeg; vt < vend; vt += 64) {
        // stage dout[vt..vt+63][0..np) and in[nb(v)][0..kp) transposed
        for (int e = threadIdx.x; e < 64 * 64; e += 256) {
            const int vl = e >> 6, c = e & 63;
            const long v = vt + vl;
            unsigned short dval = 0, ival = 0;
            if (v < vend) {
                if (c < a.nout) dval = a.dout[v * a.ldd + c];
                if (c < a.kin) ival = a.in[conv_nb(v, o, 1, g) * a.kin + c];
            }
            sd[c][vl] = dval;
            si[c][vl] = ival;
        }
        __syncthreads();
        if (32 * wn < a.np && 32 * wk < a.kp) {
#pragma unroll
            for (int k0 = 0; k0 < 64; k0 += 8) {
                bf16x4 av, bv;
                const unsigned short *pa = &sd[32 * wn + row][k0 + kh];
                const unsigned short *pb = &si[32 * wk + row][k0 + kh];
                av = bf16x4{(short)pa[0], (short)pa[1], (short)pa[2], (short)pa[3]};
                bv = bf16x4{(short)pb[0], (short)pb[1], (short)pb[2], (short)pb[3]};
                acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(av, bv, acc, 0, 0, 0);
            }
        }
        __syncthreads();
    }
    if (32 * wn < a.np && 32 * wk < a.kp) {
        const int col = 32 * wk + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int n = 32 * wn + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            a.part[(((size_t)blockIdx.x * 27 + o) * a.np + n) * a.kp + col] = acc[r];
        }
    }
}

// Weight gradient on the K = 16 MFMA, organised by x-rows: a block owns a
// range of rows (y, z, b) and one (dy, dz) pair (blockIdx.y), stages each
// row's output gradient dout[x][n] transposed as sd[n][x] and the matching
// input row at (y + dy, z + dz) as three x-shifted copies si[dx][k][x], so the
// three dx offsets are aligned 16-byte LDS reads; a wave owns up to three of
// the (n-tile, k-tile, dx) 32×32 accumulators.  Partials
// part[blockIdx.x][o][n][k] as k_conv_wgrad.  Needs M % 16 == 0, np and kp
// in {32, 64}, ldd and kin multiples of 8.  LDS 4·64·(M + 8) halves.
// Halves q of four 16-byte vectors (8 BF16 channels of 4 voxels) packed
// into one 8-byte word in voxel order: the 4×8 → 8×4 register transpose of
// the weight-gradient staging.
__device__ inline uint2 pack4_bf16(const u32x4 (&v)[4], int q)
{
    auto half = [&](const u32x4 &w) -> unsigned int {
        const unsigned int word = (q >> 1) == 0 ? w.x : (q >> 1) == 1 ? w.y : (q >> 1) == 2 ? w.z : w.w;
        return (q & 1) ? (word >> 16) : (word & 0xffffu);
    };
    return make_uint2(half(v[0]) | (half(v[1]) << 16), half(v[2]) | (half(v[3]) << 16));
}

struct WGrad16Args {
    const unsigned short *dout; // [V][ldd]
    const unsigned short *in;   // [V][kin]
    float *part;
    int ldd, nout, kin, np, kp;
    int rows_per_block;
};

__global__ void __launch_bounds__(256) k_conv_wgrad16(WGrad16Args a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    unsigned short *lds = reinterpret_cast<unsigned short *>(smem_raw);
    const int M = g.M, LD = M + 8;
    unsigned short *sd = lds;           // [64][LD]
    unsigned short *si = lds + 64 * LD; // [3][64][LD]
    const int grp = blockIdx.y, dy = grp % 3 - 1, dz = grp / 3 - 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 31, h = lane >> 5;
    const int NT = a.np / 32, KT = a.kp / 32, ntiles = NT * KT * 3;
    const int nc8 = a.np / 8, kc8 = a.kp / 8;
    f32x16 acc[3];
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
    const long nrows = (long)g.B * M * M;
    const long r0 = (long)blockIdx.x * a.rows_per_block;
    const long r1 = min(nrows, r0 + a.rows_per_block);
    const u32x4 zero4 = {0u, 0u, 0u, 0u};
    for (long r = r0; r < r1; ++r) {
        const int y = (int)(r % M);
        const long t = r / M;
        const int z = (int)(t % M);
        const long b = t / M;
        const int ys = y + dy < 0 ? y + dy + M : (y + dy >= M ? y + dy - M : y + dy);
        const int zs = z + dz < 0 ? z + dz + M : (z + dz >= M ? z + dz - M : z + dz);
        const long vrow = r * M, vsrc = (long)M * (ys + (long)M * (zs + (long)M * b));
        __syncthreads();
        // groups of 4 voxels × 8 channels are loaded as four 16-byte vectors and
        // written transposed as eight 8-byte LDS stores
        for (int e = threadIdx.x; e < (M / 4) * nc8; e += blockDim.x) {
            const int xg = e / nc8, c8 = (e - xg * nc8) * 8, x = 4 * xg;
            u32x4 v[4];
#pragma unroll
            for (int vi = 0; vi < 4; ++vi)
                v[vi] = c8 + 8 <= a.ldd ? *reinterpret_cast<const u32x4 *>(a.dout + (vrow + x + vi) * a.ldd + c8) : zero4;
#pragma unroll
            for (int q = 0; q < 8; ++q)
                *reinterpret_cast<uint2 *>(sd + (c8 + q) * LD + x) = pack4_bf16(v, q);
        }
        for (int e = threadIdx.x; e < 3 * (M / 4) * kc8; e += blockDim.x) {
            const int dxi = e / ((M / 4) * kc8), f = e - dxi * ((M / 4) * kc8);
            const int xg = f / kc8, c8 = (f - xg * kc8) * 8, x = 4 * xg;
            u32x4 v[4];
#pragma unroll
            for (int vi = 0; vi < 4; ++vi) {
                int xs = x + vi + dxi - 1; // si[dx][k][x] = in[(x + dx) mod M][k]
                xs = xs < 0 ? xs + M : (xs >= M ? xs - M : xs);
                v[vi] = c8 + 8 <= a.kin ? *reinterpret_cast<const u32x4 *>(a.in + (vsrc + xs) * a.kin + c8) : zero4;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
                *reinterpret_cast<uint2 *>(si + (dxi * 64 + c8 + q) * LD + x) = pack4_bf16(v, q);
        }
        __syncthreads();
#pragma unroll
        for (int ti = 0; ti < 3; ++ti) {
            const int tile = wave + 4 * ti;
            if (tile >= ntiles) break;
            const int dxi = tile % 3, rest = tile / 3, nt = rest % NT, kt = rest / NT;
            const unsigned short *pa = sd + (32 * nt + row) * LD + 8 * h;
            const unsigned short *pb = si + (dxi * 64 + 32 * kt + row) * LD + 8 * h;
            for (int x0 = 0; x0 < M; x0 += 16) {
                const bf16x8 av = *reinterpret_cast<const bf16x8 *>(pa + x0);
                const bf16x8 bv = *reinterpret_cast<const bf16x8 *>(pb + x0);
                acc[ti] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[ti], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int ti = 0; ti < 3; ++ti) {
        const int tile = wave + 4 * ti;
        if (tile >= ntiles) break;
        const int dxi = tile % 3, rest = tile / 3, nt = rest % NT, kt = rest / NT;
        const int o = dxi + 3 * grp;
        const int k = 32 * kt + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int n = 32 * nt + 8 * (r >> 2) + 4 * h + (r & 3);
            a.part[(((size_t)blockIdx.x * 27 + o) * a.np + n) * a.kp + k] = acc[ti][r];
        }
    }
}

// Weight gradient by x-rows with one staged input row for all three dx
// offsets.  A block owns a range of rows (y, z, b) and one (dy, dz) pair
// (blockIdx.y); per row it stages the output gradient transposed,
// sd[n][x], and the input row at (y + dy, z + dz) transposed with an
// 8-voxel periodic halo on each side, si[k][x + 8].  Wave w takes the
// 16-voxel reduction slices x0 = 16 s (s ≡ w mod 4) and accumulates every
// (n-tile, k-tile, dx) tile of the block, NT·KT·3 ≤ 12: each slice reads one
// A fragment per n-tile and, per k-tile, the aligned 16-byte chunk at x0 plus
// the neighbouring dwords, from which the dx = ±1 operands are built by
// 16-bit funnel shifts (the reduction index pairs dout[x] with in[x + dx]).
// The global loads of the next row are issued into registers before the
// current row's MFMAs, so their latency overlaps the arithmetic.  Staging
// writes 8 voxels × 8 channels per thread as eight 16-byte transposed rows;
// row strides are ≡ 4 dwords (mod 8), which keeps both the transposed
// writes (lanes along x) and the fragment reads (lanes along channels) free
// of bank conflicts.  At the end the waves' tiles are summed in LDS in wave
// order (deterministic) and written as part[blockIdx.x][o][n][k].
// Needs M % 16 == 0, M <= 64, NT = np/32 and KT = kp/32 in {1, 2}, ldd and
// kin multiples of 8.
struct WGradRowArgs {
    const unsigned short *dout; // [V][ldd]
    const unsigned short *in;   // [V][kin]
    float *part;
    int ldd, kin;
    int rows_per_block;
    int lds_d, lds_i; // row strides of sd and si in halves
};

__host__ __device__ constexpr int wgrad_row_stride(int halves)
{
    // dwords rounded up to ≡ 4 (mod 8), returned in halves
    return 2 * ((halves / 2 + 3) / 8 * 8 + 4);
}

__device__ inline unsigned int bf_pair(unsigned int a, unsigned int b, int q)
{
    // element q (0..1 inside the dword) of a and of b as (a_q | b_q << 16)
    return q ? ((a >> 16) | (b & 0xffff0000u)) : ((a & 0xffffu) | (b << 16));
}

template <int NT, int KT>
__global__ void __launch_bounds__(256) k_conv_wgrad_rows(WGradRowArgs a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    unsigned short *lds = reinterpret_cast<unsigned short *>(smem_raw);
    constexpr int NP = 32 * NT, KP = 32 * KT, NTILE = NT * KT * 3;
    const int M = g.M, LDD = a.lds_d, LDI = a.lds_i;
    unsigned short *sd = lds;            // [NP][LDD]
    unsigned short *si = lds + NP * LDD; // [KP][LDI], column x + 8
    const int grp = blockIdx.y, dy = grp % 3 - 1, dz = grp / 3 - 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 31, h = lane >> 5;
    const int MG = M / 8;                        // 8-voxel groups per row
    const int nd = MG * (NP / 8);                // staging items of dout
    const int ni = (MG + 2) * (KP / 8);          // staging items of the input (with halo)
    const long nrows = (long)g.B * M * M;
    const long r0 = (long)blockIdx.x * a.rows_per_block;
    const long r1 = min(nrows, r0 + a.rows_per_block);
    const u32x4 zero4 = {0u, 0u, 0u, 0u};

    f32x16 acc[NTILE];
#pragma unroll
    for (int t = 0; t < NTILE; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;

    // this thread's staging item (at most one of the 2 kinds; nd + ni <= 256)
    const int e = threadIdx.x;
    const bool isd = e < nd, isi = !isd && e < nd + ni;
    int xg = 0, c8 = 0;
    if (isd) {
        xg = e % MG;
        c8 = 8 * (e / MG);
    } else if (isi) {
        xg = (e - nd) % (MG + 2);
        c8 = 8 * ((e - nd) / (MG + 2));
    }
    u32x4 pf[8];
    auto fetch = [&](long r) __attribute__((always_inline)) {
        const int y = (int)(r % M);
        const long t = r / M;
        const int z = (int)(t % M);
        const long b = t / M;
        if (isd) {
            const long v0 = r * M + 8 * xg;
            const bool ok = c8 + 8 <= a.ldd;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                pf[i] = ok ? *reinterpret_cast<const u32x4 *>(a.dout + (v0 + i) * a.ldd + c8) : zero4;
        } else if (isi) {
            const int ys = y + dy < 0 ? y + dy + M : (y + dy >= M ? y + dy - M : y + dy);
            const int zs = z + dz < 0 ? z + dz + M : (z + dz >= M ? z + dz - M : z + dz);
            const long vrow = (long)M * (ys + (long)M * (zs + (long)M * b));
            int xs = 8 * xg - 8; // halo groups wrap periodically
            xs = xs < 0 ? xs + M : (xs >= M ? xs - M : xs);
            const bool ok = c8 + 8 <= a.kin;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                pf[i] = ok ? *reinterpret_cast<const u32x4 *>(a.in + (vrow + xs + i) * a.kin + c8) : zero4;
        }
    };
    auto stage = [&]() __attribute__((always_inline)) {
        if (!isd && !isi) return;
        unsigned short *dst = isd ? sd + c8 * LDD + 8 * xg : si + c8 * LDI + 8 * xg;
        const int ld = isd ? LDD : LDI;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int wq = q >> 1, hq = q & 1;
            auto w = [&](const u32x4 &v) { return wq == 0 ? v.x : wq == 1 ? v.y : wq == 2 ? v.z : v.w; };
            u32x4 o;
            o.x = bf_pair(w(pf[0]), w(pf[1]), hq);
            o.y = bf_pair(w(pf[2]), w(pf[3]), hq);
            o.z = bf_pair(w(pf[4]), w(pf[5]), hq);
            o.w = bf_pair(w(pf[6]), w(pf[7]), hq);
            *reinterpret_cast<u32x4 *>(dst + q * ld) = o;
        }
    };

    if (r0 < r1) fetch(r0);
    for (long r = r0; r < r1; ++r) {
        __syncthreads(); // the previous row's fragments are read
        stage();
        __syncthreads();
        if (r + 1 < r1) fetch(r + 1);
        for (int s = wave; s < M / 16; s += 4) {
            const int x0 = 16 * s;
            bf16x8 av[NT];
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                av[nt] = *reinterpret_cast<const bf16x8 *>(sd + (32 * nt + row) * LDD + x0 + 8 * h);
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) {
                const unsigned short *pk = si + (32 * kt + row) * LDI + 8 + x0 + 8 * h;
                const u32x4 c = *reinterpret_cast<const u32x4 *>(pk);
                const unsigned int prev = *reinterpret_cast<const unsigned int *>(pk - 2); // x - 2, x - 1
                const unsigned int next = *reinterpret_cast<const unsigned int *>(pk + 8); // x + 8, x + 9
                const unsigned int s01 = __builtin_amdgcn_alignbit(c.y, c.x, 16);
                const unsigned int s12 = __builtin_amdgcn_alignbit(c.z, c.y, 16);
                const unsigned int s23 = __builtin_amdgcn_alignbit(c.w, c.z, 16);
                const u32x4 bm = {__builtin_amdgcn_alignbit(c.x, prev, 16), s01, s12, s23}; // in[x − 1]
                const u32x4 bp = {s01, s12, s23, __builtin_amdgcn_alignbit(next, c.w, 16)}; // in[x + 1]
                const bf16x8 bv[3] = {__builtin_bit_cast(bf16x8, bm), __builtin_bit_cast(bf16x8, c),
                                      __builtin_bit_cast(bf16x8, bp)};
#pragma unroll
                for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                    for (int dxi = 0; dxi < 3; ++dxi) {
                        f32x16 &ac = acc[(nt * KT + kt) * 3 + dxi];
                        ac = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[nt], bv[dxi], ac, 0, 0, 0);
                    }
            }
        }
    }
    // ordered sum of the waves' tiles in LDS, then the block's partials
    float *red = reinterpret_cast<float *>(smem_raw);
    __syncthreads();
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int t = 0; t < NTILE; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int idx = t * 1024 + (8 * (r >> 2) + 4 * h + (r & 3)) * 32 + row;
                    red[idx] = w == 0 ? acc[t][r] : red[idx] + acc[t][r];
                }
        }
        __syncthreads();
    }
    for (int idx = threadIdx.x; idx < NTILE * 1024; idx += blockDim.x) {
        const int t = idx >> 10, i = (idx >> 5) & 31, j = idx & 31;
        const int dxi = t % 3, kt = (t / 3) % KT, nt = t / (3 * KT);
        const int o = dxi + 3 * grp;
        a.part[(((size_t)blockIdx.x * 27 + o) * NP + 32 * nt + i) * KP + 32 * kt + j] = red[idx];
    }
}

// Weight gradient by x-rows, one dz per block (blockIdx.y): the block walks a
// contiguous range of rows r = y + M (z + M b) and accumulates the nine
// (dy, dx) offsets of its dz at once.  Rows sit in LDS as they do in HBM
// (voxel by voxel, channels contiguous) and the MFMA operands, which need
// eight consecutive voxels of one channel per lane, come from
// ds_read_b64_tr_b16 (each 16-lane group reads 4 voxels × 16 channels and
// receives them transposed); the dx = ±1 operands are the same reads one
// voxel on.  So staging is a copy (the earlier kernel transposed 8 × 8
// tiles in registers and built the shifted operands from two conflicting
// 4-byte reads and seven funnel shifts each: 1.79 ms per 64 → 64 layer of a
// 16 × 64³ batch, 23 % MFMA busy).
//
// LDS: two output-gradient rows (the next one is written while the current
// one is read) and a ring of four input rows y−1 … y+2 (row y' in slot
// (y' + 1) mod 4) with one halo voxel on each side, so a row costs one
// barrier; its global loads are in flight during the MFMAs of the two rows
// before (one row ahead left the kernel waiting on them: 1.30 ms per 64 → 64
// layer, two 0.97–1.02; 3 → 64 0.61 and 64 → 6 0.51, from 1.66 and 1.33).
// 64-channel rows (128 bytes) swap their 64-byte halves on every
// second pair of voxels: the 4 voxels × 64 bytes that 32 lanes read then
// cover all banks once.
//
// Wave w takes the (n-tile, k-tile) pair w mod NT·KT and the 16-voxel slices
// s ≡ w / (NT·KT) (mod 4 / (NT·KT)); waves sharing a pair write partials of
// their own: part[blockIdx.x · WPC + w / (NT·KT)][o][n][k].
// Rows of M % 16 != 0 voxels are filled up to MP with zeros; two training
// steps against the voxel-tile kernel (k_conv_wgrad): 16 × 8³ 0.66 / 5.9 ms,
// 4 × 24³ 0.87 / 6.7, 12 × 40³ 4.1 / 34.7.
//
// FOLD: the narrow operand of the first and last layers (3 input or 6 output
// channels, at most 8) is staged three times, shifted by dx, as 24 of 32
// channels, so one MFMA covers the three dx (FOLD = 1: output gradient,
// E[x][8 d + n] = dout[x − (d − 1)][n]; FOLD = 2: input, E[x][8 d + c] =
// in[x + d − 1][c]) and the nine accumulators become three (16 × 64³: 64 → 6
// 579 -> 396 µs, 3 → 64 492 -> 278; barriers and load latency per row are what
// is left).
// Needs M <= 64 (two 16-byte pieces of a row per thread), NT = np/32 and KT = kp/32 in {1, 2}, ldd and
// kin multiples of 8.
struct WGradTrArgs {
    const unsigned short *dout; // [V][ldd]
    const unsigned short *in;   // [V][kin]
    float *part;
    float *bpart; // bias-gradient partials bpart[c · gridDim.x + blockIdx.x] (dz = 0 blocks)
    int nout;
    int ldd, kin;
    int rows_per_block;
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bf16x8 lds_read_tr(const unsigned char *p, int second)
{
    typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
    struct pair {
        i16x4 a, b;
    } v;
    v.a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)p);
    v.b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + second));
    return __builtin_bit_cast(bf16x8, v);
}

template <int NT, int KT, int FOLD>
__global__ void __launch_bounds__(256, FOLD ? 3 : 2) k_conv_wgrad_tr(WGradTrArgs a, ConvGeom g)
{
    extern __shared__ unsigned char smem_raw[];
    constexpr int NP = 32 * NT, KP = 32 * KT, NC = NT * KT, WPC = 4 / NC;
    constexpr int RD = 2 * NP, RI = 2 * KP; // bytes per voxel of the two row kinds
    constexpr int PMAX = 2;                 // 16-byte pieces of a row per thread (M <= 64)
    constexpr int PD = FOLD == 1 ? 1 : PMAX, PI = FOLD == 2 ? 1 : PMAX, NA = FOLD ? 3 : 9;
    static_assert(FOLD == 0 || (FOLD == 1 ? NT == 1 : KT == 1), "the folded operand has one tile");
    const int M = g.M, MP = (M + 15) & ~15, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    unsigned char *sd = smem_raw;                // [2][MP][NP]
    unsigned char *si = smem_raw + 2 * MP * RD;  // [4][MP + 2][KP], voxel x at x + 1
    const int SLOT = (MP + 2) * RI;
    const int dzi = blockIdx.y;
    const int combo = wave % NC, sg = wave / NC, nt = combo % NT, kt = combo / NT;
    const int nrows = g.B * M * M;
    const int r0 = blockIdx.x * a.rows_per_block, r1 = min(nrows, r0 + a.rows_per_block);

    // byte of (voxel, channel byte) in a row of CB bytes per voxel
    auto at = [](int v, int cb, int CB) { return v * CB + (CB == 128 ? cb ^ (((v >> 1) & 1) << 6) : cb); };

    // lane offsets of the transposed reads: 16-lane group (channel half,
    // voxel half), voxel i / 4 and channels 4 (i mod 4) .. +3 within it
    const int i16 = lane & 15, ch = 16 * ((lane >> 4) & 1) + 4 * (i16 & 3), vx = 8 * (lane >> 5) + (i16 >> 2);
    const int offa = at(vx, 2 * (32 * nt + ch), RD);
    int offb[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) offb[d] = at(vx + d, 2 * (32 * kt + ch), RI);

    // row pieces: piece e is 8 channels (16 bytes) of voxel e / (channels / 8)
    // (of a folded operand only the first 8 channels)
    const int pcd = FOLD == 1 ? 1 : a.ldd / 8, pci = FOLD == 2 ? 1 : a.kin / 8, nd = M * pcd, ni = M * pci;
    const int stepd = FOLD == 1 ? a.ldd : 8, stepi = FOLD == 2 ? a.kin : 8; // halves between pieces
    // the three places of a folded voxel's channels
    auto store3 = [&](unsigned char *p, int v, int dir, const u32x4 &w) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int x = v + dir * (d - 1);
            x = x < 0 ? M - 1 : x >= M ? 0 : x;
            *reinterpret_cast<u32x4 *>(p + 64 * x + 16 * d) = w;
        }
    };
    float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const bool dobias = dzi == 1;
    // (pieces past the row read its last one again: no branch around the
    // loads, so the waits for one row's pieces leave the next row's in flight)
    auto load_d = [&](u32x4 (&pd)[PD], int r) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < PD; ++q)
            pd[q] = *reinterpret_cast<const u32x4 *>(a.dout + ((size_t)r * nd + min(tid + 256 * q, nd - 1)) * stepd);
    };
    auto store_d = [&](const u32x4 (&pd)[PD], int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < PD; ++q) {
            const int e = tid + 256 * q;
            if (e >= nd) continue;
            const int v = e / pcd, c = e - v * pcd;
            if constexpr (FOLD == 1) store3(sd + buf * MP * RD, v, 1, pd[q]);
            else *reinterpret_cast<u32x4 *>(sd + buf * MP * RD + at(v, 16 * c, RD)) = pd[q];
            if (dobias) {
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    bsum[2 * w] += bf2f((unsigned short)(pd[q][w] & 0xffffu));
                    bsum[2 * w + 1] += bf2f((unsigned short)(pd[q][w] >> 16));
                }
            }
        }
    };
    // input row yin (−1 … M) of plane z + dz of the sample of plane p
    auto load_i = [&](u32x4 (&pi)[PI], int p, int yin) __attribute__((always_inline)) {
        const int z = p % M, zs = z + dzi - 1, zw = zs < 0 ? zs + M : zs >= M ? zs - M : zs;
        const int yw = yin < 0 ? yin + M : yin >= M ? yin - M : yin;
        const size_t row = (size_t)(p - z + zw) * M + yw;
#pragma unroll
        for (int q = 0; q < PI; ++q)
            pi[q] = *reinterpret_cast<const u32x4 *>(a.in + (row * ni + min(tid + 256 * q, ni - 1)) * stepi);
    };
    auto store_i = [&](const u32x4 (&pi)[PI], int yin) __attribute__((always_inline)) {
        unsigned char *slot = si + ((yin + 1) & 3) * SLOT;
#pragma unroll
        for (int q = 0; q < PI; ++q) {
            const int e = tid + 256 * q;
            if (e >= ni) continue;
            const int v = e / pci, c = e - v * pci;
            if constexpr (FOLD == 2) {
                store3(slot + RI, v, -1, pi[q]);
                continue;
            }
            *reinterpret_cast<u32x4 *>(slot + at(v + 1, 16 * c, RI)) = pi[q];
            // the periodic halo: voxel 0 again behind the row, voxel M−1 before it
            if (v == 0) *reinterpret_cast<u32x4 *>(slot + at(M + 1, 16 * c, RI)) = pi[q];
            if (v == M - 1) *reinterpret_cast<u32x4 *>(slot + at(0, 16 * c, RI)) = pi[q];
        }
    };

    // channels past ldd and kin and voxels past M stay zero
    if (a.ldd < NP || a.kin < KP || MP != M)
        for (int e = tid; e < (2 * MP * RD + 4 * SLOT) / 16; e += 256)
            reinterpret_cast<u32x4 *>(smem_raw)[e] = u32x4{0u, 0u, 0u, 0u};

    f32x16 acc[NA];
#pragma unroll
    for (int t = 0; t < NA; ++t)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[t][q] = 0.0f;

    // one row: LDS holds its output gradient and input rows y−1 … y+1, (pd, pi)
    // the next output-gradient row and input row y+2 (in flight since the
    // row before), (qd, qi) receive those of the row after
    auto row_step = [&](u32x4 (&pd)[PD], u32x4 (&pi)[PI], u32x4 (&qd)[PD], u32x4 (&qi)[PI], int p, int y, int y1,
                        int cur) __attribute__((always_inline)) {
        const int yn = min(y + 2, y1 - 1); // rows past the range: loaded, not stored
        load_d(qd, p * M + yn);
        load_i(qi, p, yn + 1);
        const unsigned char *da = sd + cur * MP * RD + offa;
        for (int s = sg; s < MP / 16; s += WPC) {
            const bf16x8 av = lds_read_tr(da + 16 * s * RD, 4 * RD);
#pragma unroll
            for (int dyi = 0; dyi < 3; ++dyi) {
                const unsigned char *bi = si + ((y + dyi) & 3) * SLOT + 16 * s * RI; // row y + dyi − 1
                if constexpr (FOLD != 0) {
                    acc[dyi] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, lds_read_tr(bi + offb[1], 4 * RI), acc[dyi], 0, 0, 0);
                    continue;
                }
                bf16x8 bv[3];
#pragma unroll
                for (int d = 0; d < 3; ++d) bv[d] = lds_read_tr(bi + offb[d], 4 * RI);
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    acc[3 * dyi + d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv[d], acc[3 * dyi + d], 0, 0, 0);
            }
        }
        if (y + 1 < y1) {
            store_d(pd, cur ^ 1);
            store_i(pi, y + 2);
        }
        __syncthreads();
    };
    for (int r = r0; r < r1;) {
        // the rows of one plane
        const int p = r / M, y0 = r - p * M, y1 = min(M, y0 + r1 - r);
        u32x4 pd[PD], pi[PI], qd[PD], qi[PI], ri[PI];
        __syncthreads();
        load_d(pd, r);
        load_i(pi, p, y0 - 1);
        load_i(qi, p, y0);
        load_i(ri, p, y0 + 1);
        store_d(pd, 0);
        store_i(pi, y0 - 1);
        store_i(qi, y0);
        store_i(ri, y0 + 1);
        load_d(pd, p * M + min(y0 + 1, y1 - 1));
        load_i(pi, p, min(y0 + 2, M));
        __syncthreads();
        for (int y = y0; y < y1; y += 2) {
            row_step(pd, pi, qd, qi, p, y, y1, (y - y0) & 1);
            if (y + 1 < y1) row_step(qd, qi, pd, pi, p, y + 1, y1, (y + 1 - y0) & 1);
        }
        r += y1 - y0;
    }
    if (dobias) {
        // threads tid ≡ c (mod pcd) hold the channels 8 c .. 8 c + 7
        float *red = reinterpret_cast<float *>(smem_raw);
#pragma unroll
        for (int q = 0; q < 8; ++q) red[tid * 8 + q] = bsum[q];
        __syncthreads();
        if (tid < 8 * pcd && tid < a.nout) {
            float t = 0.f;
            for (int x = tid / 8; x < 256; x += pcd) t += red[x * 8 + (tid & 7)];
            a.bpart[(size_t)tid * gridDim.x + blockIdx.x] = t;
        }
    }
    const size_t pbase = ((size_t)blockIdx.x * WPC + sg) * 27 + 9 * dzi;
    const int row = lane & 31, h = lane >> 5;
#pragma unroll
    for (int t = 0; t < NA; ++t)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int i = 8 * (q >> 2) + 4 * h + (q & 3);
            if constexpr (FOLD == 0) {
                a.part[((pbase + t) * NP + 32 * nt + i) * KP + 32 * kt + row] = acc[t][q];
            } else if constexpr (FOLD == 1) { // row i = 8 dx + n
                if (q < 12) a.part[((pbase + 3 * t + (q >> 2)) * NP + (i & 7)) * KP + 32 * kt + row] = acc[t][q];
            } else { // column 8 dx + c
                if (row < 24) a.part[((pbase + 3 * t + (row >> 3)) * NP + 32 * nt + i) * KP + (row & 7)] = acc[t][q];
            }
        }
}

// Sums the partials over the voxel splits into the FP32 gradient
// grad[o][n][k] (n < nout, k < kin) of the unpadded layout.  A block takes 64
// consecutive elements; its four wavefronts sum the splits q ≡ wave (mod 4) in
// order, eight loads in flight each, and the four sums are added pairwise
// (fixed order).  One thread per element with four loads in flight left the
// reads latency-bound: 29-43 µs per layer for 170 splits, 75 MB.
// The nout blocks past those sum the bias partials bpart[c][x], x < nb, one
// channel each: strided FP64 partial sums, then a tree in LDS (a launch of its
// own took 4.8 µs per layer).
__global__ void __launch_bounds__(256) k_wgrad_reduce(const float *part, int nsplit, int np, int kp, int nout, int kin,
                                                      float *grad, const float *bpart, int nb, float *bgrad)
{
    __shared__ double s[4][64];
    const int wblocks = (27 * nout * kin + 63) / 64;
    if ((int)blockIdx.x >= wblocks) {
        const int c = blockIdx.x - wblocks;
        double *sb = s[0];
        double acc = 0;
        for (int q = threadIdx.x; q < nb; q += blockDim.x) acc += bpart[(size_t)c * nb + q];
        sb[threadIdx.x] = acc;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (threadIdx.x < w) sb[threadIdx.x] += sb[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) bgrad[c] = (float)sb[0];
        return;
    }
    const int total = 27 * nout * kin, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t = blockIdx.x * 64 + lane, tc = min(t, total - 1);
    const int k = tc % kin, n = (tc / kin) % nout, o = tc / (kin * nout);
    const size_t stride = (size_t)27 * np * kp;
    const float *src = part + ((size_t)o * np + n) * kp + k;
    double acc = 0;
    int q = wave;
    for (; q + 28 < nsplit; q += 32) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = src[(size_t)(q + 4 * e) * stride];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += v[e];
    }
    for (; q < nsplit; q += 4) acc += src[(size_t)q * stride];
    s[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && t < total) grad[t] = (float)((s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]));
}

// Bias gradient: per-channel sum of dout over all voxels (per-block
// partials part[c · gridDim + block]).  A thread reads 8 channels (16 bytes)
// of a voxel row, ldd/8 threads cover a row and a block 256·8/ldd rows per
// pass, so waves read contiguous channel-last memory, dout is read once and
// each load moves 16 bytes (ldd a multiple of 8 dividing 2048).  1D grid.
__global__ void __launch_bounds__(256) k_bias_grad(const unsigned short *dout, int ldd, int nout, long V, float *part)
{
    __shared__ float s[8][256];
    const int tpr = ldd / 8, c8 = threadIdx.x % tpr, r = threadIdx.x / tpr, rows = blockDim.x / tpr;
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll 4
    for (long v = blockIdx.x * (long)rows + r; v < V; v += (long)gridDim.x * rows) {
        const uint4 q = *reinterpret_cast<const uint4 *>(dout + v * ldd + 8 * c8);
        const unsigned int w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[2 * e] += bf2f((unsigned short)(w[e] & 0xffffu));
            acc[2 * e + 1] += bf2f((unsigned short)(w[e] >> 16));
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) s[e][threadIdx.x] = acc[e];
    __syncthreads();
    // thread (row 0, c8) sums its 8 channels over the block's rows
    if (r == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = 8 * c8 + e;
            if (c >= nout) continue;
            float t = 0;
            for (int q = 0; q < rows; ++q) t += s[e][q * tpr + c8];
            part[(size_t)c * gridDim.x + blockIdx.x] = t;
        }
    }
}

// MSE loss over `nout` channels: dy = 2(y − t)/(V nout) (BF16, padded to
// ldd channels with zeros), per-block partial sums of (y − t)².
__global__ void __launch_bounds__(256) k_mse(const float *y, const float *t, int nout, long V, unsigned short *dy,
                                             int ldd, double *part)
{
    // one voxel per thread and pass: the ldd BF16 gradient channels (zero
    // past nout) leave as 16-byte stores of 8 channels (ldd % 8 == 0)
    __shared__ double s[256];
    const double scale = 2.0 / ((double)V * nout);
    double acc = 0;
    for (long v = blockIdx.x * (long)blockDim.x + threadIdx.x; v < V; v += (long)gridDim.x * blockDim.x) {
        for (int c0 = 0; c0 < ldd; c0 += 8) {
            unsigned int w[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                unsigned short hb[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int c = c0 + 2 * q + e;
                    float d = 0.f;
                    if (c < nout) {
                        const float r = y[v * nout + c] - t[v * nout + c];
                        acc += (double)r * r;
                        d = (float)(scale * r);
                    }
                    hb[e] = f2bf(d);
                }
                w[q] = (unsigned int)hb[0] | ((unsigned int)hb[1] << 16);
            }
            *reinterpret_cast<u32x4 *>(dy + v * ldd + c0) = u32x4{w[0], w[1], w[2], w[3]};
        }
    }
    s[threadIdx.x] = acc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// Adam on FP32 masters; refreshes the BF16 forward (W[o][n][k], n padded to
// np) and transposed (WT[o][k][n], k padded to kpt) copies in the same pass
// (their padding stays as k_pack_weights wrote it; a pack launch per layer
// took 27 µs of a 475 µs step of 4 × 32³).  The bias tail of each layer is
// stored after its weights in the flat parameter vector.
struct AdamLayer {
    int woff, nw; // weights of the layer in the flat vector: [woff, woff + nw), order [o][n][k]
    int nout, kin, np, kinp, kpt, noutp;
    unsigned short *W, *WT;
};
struct AdamArgs {
    float *w, *m, *v;
    const float *g;
    int count;
    float lr, b1, b2, eps, c1, c2; // c1 = 1/(1−b1^t), c2 = 1/(1−b2^t)
    AdamLayer layer[4];
};

__global__ void __launch_bounds__(256) k_adam(AdamArgs a)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.count) return;
    const float g = a.g[t];
    const float m = a.b1 * a.m[t] + (1.f - a.b1) * g;
    const float v = a.b2 * a.v[t] + (1.f - a.b2) * g * g;
    a.m[t] = m;
    a.v[t] = v;
    const float mh = m * a.c1, vh = v * a.c2;
    const float w = a.w[t] - a.lr * mh / (sqrtf(vh) + a.eps);
    a.w[t] = w;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const AdamLayer &c = a.layer[l];
        const int e = t - c.woff;
        if (e < 0 || e >= c.nw) continue;
        const int k = e % c.kin, n = (e / c.kin) % c.nout, o = e / (c.kin * c.nout);
        const unsigned short h = f2bf(w);
        c.W[(o * c.np + n) * c.kinp + k] = h;
        c.WT[(o * c.kpt + k) * c.noutp + n] = h;
    }
}

// Writes the BF16 copies of one layer's weights from its FP32 master w[o][n][k]
// (n < nout, k < kin): W[o][n][k] with n padded to np and k to kinp, and
// WT[o][k][n] with k padded to kpt (rows) and n to noutp (contiguous).
__global__ void k_pack_weights(const float *w, int nout, int kin, unsigned short *W, int np, int kinp,
                               unsigned short *WT, int kpt, int noutp)
{
    const int total = 27 * np * kinp;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += gridDim.x * blockDim.x) {
        const int k = t % kinp, n = (t / kinp) % np, o = t / (kinp * np);
        const float val = (n < nout && k < kin) ? w[(o * nout + n) * kin + k] : 0.f;
        W[t] = f2bf(val);
    }
    if (!WT) return;
    const int totalT = 27 * kpt * noutp;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < totalT; t += gridDim.x * blockDim.x) {
        const int n = t % noutp, k = (t / noutp) % kpt, o = t / (noutp * kpt);
        const float val = (n < nout && k < kin) ? w[(o * nout + n) * kin + k] : 0.f;
        WT[t] = f2bf(val);
    }
}

// FP32 planar (V, cin) → BF16 channels-last padded to ldc channels, with a
// scale; and the inverse for FP32 outputs.
__global__ void k_to_bf16(const float *x, int cin, float scale, long V, unsigned short *out, int ldc)
{
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < V * ldc; e += (long)gridDim.x * blockDim.x) {
        const long v = e / ldc;
        const int c = (int)(e - v * ldc);
        out[e] = c < cin ? f2bf(scale * x[v * cin + c]) : (unsigned short)0;
    }
}

}  // namespace dns
