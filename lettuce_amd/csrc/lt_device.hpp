// lt_device.hpp -- device-side building blocks for the gfx950 gauge-field kernels:
// FP64 complex and 3x3 matrix arithmetic, the even/odd structure-of-arrays link
// layout, lattice neighbour arithmetic, the Philox4x32-10 counter RNG, SU(2)
// subgroup helpers, Gram-Schmidt reunitarisation and the Cayley-Hamilton
// exponential.  Everything here is FP64 VALU code; MFMA is not used because a
// 3x3 complex product is not a dense contraction worth tiling.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Launch-shape knobs of the link-update kernels (sweeps, stout, flow stages).
// LT_LINK_BS is the largest thread block they are compiled for; the host never
// launches them with more threads (tiles are validated against it).
#ifndef LT_LINK_BS
#define LT_LINK_BS 256
#endif
#ifndef LT_LINK_WAVES
#define LT_LINK_WAVES 2
#endif
#ifndef LT_XCD_REMAP
#define LT_XCD_REMAP 1
#endif
// order the t tiles of each XCD's block range fastest (LinkMap::tc)
#ifndef LT_TCHUNK
#define LT_TCHUNK 1
#endif
// y tiles per chunk (LinkMap::yc; 0: all y tiles in one chunk).  Two y tiles per
// chunk at 32^4 (8 tiles in flight per x step in each XCD): RK3 flow step -1 % against
// one chunk; one y tile per chunk is slower.
#ifndef LT_YCHUNK
#define LT_YCHUNK 2
#endif
#define LT_LINK_KERNEL __launch_bounds__(LT_LINK_BS) __attribute__((amdgpu_waves_per_eu(LT_LINK_WAVES)))

namespace lt {

// Workgroups are dispatched round-robin over the 8 XCDs of the MI355X, each with
// its own L2.  Remapping the block index so that every XCD works on one
// contiguous range of sites keeps the z/y neighbours of a block in the same L2.
__device__ __forceinline__ int xcd_block(int b, int nb)
{
#if LT_XCD_REMAP
    if ((nb & 7) == 0) return (b & 7) * (nb >> 3) + (b >> 3);
#endif
    return b;
}
// The same with each XCD's range walked backwards when rev is set.  Consecutive
// launches over the same links alternate direction, so each starts on the links
// the previous one touched last (still in the L2 and the memory-side cache).
__device__ __forceinline__ int xcd_block_dir(int b, int nb, int rev)
{
#if LT_XCD_REMAP
    if ((nb & 7) == 0) {
        const int per = nb >> 3, loc = b >> 3;
        return (b & 7) * per + (rev ? per - 1 - loc : loc);
    }
#endif
    return rev ? nb - 1 - b : b;
}

// ---------------------------------------------------------------------------
// complex double
struct cd {
    double re, im;
};

__device__ __forceinline__ cd mk(double r, double i) { return cd{r, i}; }
__device__ __forceinline__ cd operator+(cd a, cd b) { return cd{a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cd operator-(cd a, cd b) { return cd{a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cd operator-(cd a) { return cd{-a.re, -a.im}; }
__device__ __forceinline__ cd operator*(cd a, cd b)
{
    return cd{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ cd operator*(double s, cd a) { return cd{s * a.re, s * a.im}; }
__device__ __forceinline__ cd operator*(cd a, double s) { return cd{s * a.re, s * a.im}; }
__device__ __forceinline__ cd conj(cd a) { return cd{a.re, -a.im}; }
__device__ __forceinline__ cd mul_i(cd a) { return cd{-a.im, a.re}; }
__device__ __forceinline__ cd& operator+=(cd& a, cd b) { a.re += b.re; a.im += b.im; return a; }
__device__ __forceinline__ cd& operator-=(cd& a, cd b) { a.re -= b.re; a.im -= b.im; return a; }
// a * conj(b)
__device__ __forceinline__ cd mul_c(cd a, cd b)
{
    return cd{a.re * b.re + a.im * b.im, a.im * b.re - a.re * b.im};
}
// conj(a) * b
__device__ __forceinline__ cd cmul(cd a, cd b)
{
    return cd{a.re * b.re + a.im * b.im, a.re * b.im - a.im * b.re};
}
// conj(x * y - z * w) as two chains of fused multiply-adds (the third row of an
// SU(3) matrix from its first two rows)
__device__ __forceinline__ cd conj_cross(cd x, cd y, cd z, cd w)
{
    double re = z.im * w.im;
    re = fma(-z.re, w.re, re);
    re = fma(-x.im, y.im, re);
    re = fma(x.re, y.re, re);
    double im = z.im * w.re;
    im = fma(z.re, w.im, im);
    im = fma(-x.im, y.re, im);
    im = fma(-x.re, y.im, im);
    return cd{re, im};
}

// ---------------------------------------------------------------------------
// 3x3 complex matrix, row-major
struct M3 {
    cd m[9];
};

__device__ __forceinline__ M3 m3_zero()
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = cd{0.0, 0.0};
    return r;
}
__device__ __forceinline__ M3 m3_id()
{
    M3 r = m3_zero();
    r.m[0].re = r.m[4].re = r.m[8].re = 1.0;
    return r;
}
// sum_k op(a_k) op(b_k) over three complex pairs as two chains of one multiply
// and five fused multiply-adds (op = conj where CA / CB is set): 12 FP64
// instructions per complex entry instead of 16 for separate products and sums.
template <bool CA, bool CB>
__device__ __forceinline__ cd dot3(cd a0, cd b0, cd a1, cd b1, cd a2, cd b2)
{
    // (x.re + i sx x.im)(y.re + i sy y.im): re = x.re y.re - sx sy x.im y.im, im = sy x.re y.im + sx x.im y.re
    constexpr double sa = CA ? -1.0 : 1.0, sb = CB ? -1.0 : 1.0, sab = -sa * sb;
    double re = a0.re * b0.re;
    re = fma(sab * a0.im, b0.im, re);
    re = fma(a1.re, b1.re, re);
    re = fma(sab * a1.im, b1.im, re);
    re = fma(a2.re, b2.re, re);
    re = fma(sab * a2.im, b2.im, re);
    double im = (sb * a0.re) * b0.im;
    im = fma(sa * a0.im, b0.re, im);
    im = fma(sb * a1.re, b1.im, im);
    im = fma(sa * a1.im, b1.re, im);
    im = fma(sb * a2.re, b2.im, im);
    im = fma(sa * a2.im, b2.re, im);
    return cd{re, im};
}
// acc + sum_k op(a_k) op(b_k): the same chains started from acc (6 FMAs per part)
template <bool CA, bool CB>
__device__ __forceinline__ cd dot3_acc(cd acc, cd a0, cd b0, cd a1, cd b1, cd a2, cd b2)
{
    constexpr double sa = CA ? -1.0 : 1.0, sb = CB ? -1.0 : 1.0, sab = -sa * sb;
    double re = fma(a0.re, b0.re, acc.re);
    re = fma(sab * a0.im, b0.im, re);
    re = fma(a1.re, b1.re, re);
    re = fma(sab * a1.im, b1.im, re);
    re = fma(a2.re, b2.re, re);
    re = fma(sab * a2.im, b2.im, re);
    double im = fma(sb * a0.re, b0.im, acc.im);
    im = fma(sa * a0.im, b0.re, im);
    im = fma(sb * a1.re, b1.im, im);
    im = fma(sa * a1.im, b1.re, im);
    im = fma(sb * a2.re, b2.im, im);
    im = fma(sa * a2.im, b2.re, im);
    return cd{re, im};
}
// acc += a * b
__device__ __forceinline__ void mul_acc(M3& acc, const M3& a, const M3& b)
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            acc.m[3 * i + j] = dot3_acc<false, false>(acc.m[3 * i + j], a.m[3 * i], b.m[j], a.m[3 * i + 1], b.m[3 + j],
                                                      a.m[3 * i + 2], b.m[6 + j]);
}
// acc += a * b^+
__device__ __forceinline__ void mul_nd_acc(M3& acc, const M3& a, const M3& b)
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            acc.m[3 * i + j] = dot3_acc<false, true>(acc.m[3 * i + j], a.m[3 * i], b.m[3 * j], a.m[3 * i + 1],
                                                     b.m[3 * j + 1], a.m[3 * i + 2], b.m[3 * j + 2]);
}
// acc += a^+ * b
__device__ __forceinline__ void mul_dn_acc(M3& acc, const M3& a, const M3& b)
{
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            acc.m[3 * i + j] = dot3_acc<true, false>(acc.m[3 * i + j], a.m[i], b.m[j], a.m[3 + i], b.m[3 + j],
                                                     a.m[6 + i], b.m[6 + j]);
}
// a * b
__device__ __forceinline__ M3 mul(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<false, false>(a.m[3 * i], b.m[j], a.m[3 * i + 1], b.m[3 + j], a.m[3 * i + 2], b.m[6 + j]);
    return r;
}
// a * b^+
__device__ __forceinline__ M3 mul_nd(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<false, true>(a.m[3 * i], b.m[3 * j], a.m[3 * i + 1], b.m[3 * j + 1], a.m[3 * i + 2],
                                               b.m[3 * j + 2]);
    return r;
}
// a^+ * b
__device__ __forceinline__ M3 mul_dn(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<true, false>(a.m[i], b.m[j], a.m[3 + i], b.m[3 + j], a.m[6 + i], b.m[6 + j]);
    return r;
}
// Rows 0 and 1 of a * b and of a * b^+ (row 2 of a is not read; row 2 of the
// result is zero), for SU(3) products whose row 2 is rebuilt by third_row.
__device__ __forceinline__ M3 mul_r01(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<false, false>(a.m[3 * i], b.m[j], a.m[3 * i + 1], b.m[3 + j], a.m[3 * i + 2], b.m[6 + j]);
    r.m[6] = r.m[7] = r.m[8] = cd{0.0, 0.0};
    return r;
}
__device__ __forceinline__ M3 mul_nd_r01(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<false, true>(a.m[3 * i], b.m[3 * j], a.m[3 * i + 1], b.m[3 * j + 1], a.m[3 * i + 2],
                                               b.m[3 * j + 2]);
    r.m[6] = r.m[7] = r.m[8] = cd{0.0, 0.0};
    return r;
}
// rows 0 and 1 of a^+ b and of a^+ b^+ (a, b complete)
__device__ __forceinline__ M3 mul_dn_r01(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<true, false>(a.m[i], b.m[j], a.m[3 + i], b.m[3 + j], a.m[6 + i], b.m[6 + j]);
    r.m[6] = r.m[7] = r.m[8] = cd{0.0, 0.0};
    return r;
}
__device__ __forceinline__ M3 mul_dd_r01(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r.m[3 * i + j] = dot3<true, true>(a.m[i], b.m[3 * j], a.m[3 + i], b.m[3 * j + 1], a.m[6 + i], b.m[3 * j + 2]);
    r.m[6] = r.m[7] = r.m[8] = cd{0.0, 0.0};
    return r;
}
__device__ __forceinline__ M3 dag(const M3& a)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) r.m[3 * i + j] = conj(a.m[3 * j + i]);
    return r;
}
__device__ __forceinline__ M3 add(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = a.m[i] + b.m[i];
    return r;
}
__device__ __forceinline__ M3 sub(const M3& a, const M3& b)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = a.m[i] - b.m[i];
    return r;
}
__device__ __forceinline__ void acc(M3& a, const M3& b)
{
#pragma unroll
    for (int i = 0; i < 9; ++i) a.m[i] += b.m[i];
}
__device__ __forceinline__ M3 scale(double s, const M3& a)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = s * a.m[i];
    return r;
}
__device__ __forceinline__ M3 scale(cd s, const M3& a)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = s * a.m[i];
    return r;
}
__device__ __forceinline__ cd trace(const M3& a) { return a.m[0] + a.m[4] + a.m[8]; }
// Re tr(a b)
__device__ __forceinline__ double retr_mul(const M3& a, const M3& b)
{
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) s += a.m[3 * i + k].re * b.m[3 * k + i].re - a.m[3 * i + k].im * b.m[3 * k + i].im;
    return s;
}
// Re tr(a b^+) for a, b in SU(3) given by rows 0 and 1: with G_ij = row_i(a) . conj(row_j(b))
// (i, j < 2) the row-2 term conj(a_0 x a_1) . (b_0 x b_1) equals conj(G_00 G_11 - G_01 G_10)
// (Binet-Cauchy), so Re tr(a b^+) = Re(G_00 + G_11 + G_00 G_11 - G_01 G_10).
__device__ __forceinline__ double retr_su3_nd_r01(const M3& a, const M3& b)
{
    cd G[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            G[i][j] = dot3_acc<false, true>(cd{0.0, 0.0}, a.m[3 * i], b.m[3 * j], a.m[3 * i + 1], b.m[3 * j + 1],
                                            a.m[3 * i + 2], b.m[3 * j + 2]);
    const cd d = G[0][0] * G[1][1] - G[0][1] * G[1][0];
    return G[0][0].re + G[1][1].re + d.re;
}
// traceless anti-hermitian part: 1/2 (A - A^+) - 1/6 tr(A - A^+)
__device__ __forceinline__ M3 algebra(const M3& a)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) r.m[3 * i + j] = 0.5 * (a.m[3 * i + j] - conj(a.m[3 * j + i]));
    // tr(A - A^+) = 2i * sum Im A_ii
    double t = (2.0 * (a.m[0].im + a.m[4].im + a.m[8].im)) * (1.0 / 6.0);
    r.m[0].im -= t;
    r.m[4].im -= t;
    r.m[8].im -= t;
    return r;
}
// traceless hermitian part: 1/2 (A + A^+) - 1/6 tr(A + A^+)
__device__ __forceinline__ M3 tl_herm(const M3& a)
{
    M3 r;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) r.m[3 * i + j] = 0.5 * (a.m[3 * i + j] + conj(a.m[3 * j + i]));
    double t = (2.0 * (a.m[0].re + a.m[4].re + a.m[8].re)) * (1.0 / 6.0);
    r.m[0].re -= t;
    r.m[4].re -= t;
    r.m[8].re -= t;
    return r;
}

// Normalise row 0, orthogonalise and normalise row 1, row 2 = conj(row0 x row1)
__device__ __forceinline__ void gram_schmidt(M3& a)
{
    cd* m = a.m;
    double n0 = 1.0 / sqrt(m[0].re * m[0].re + m[0].im * m[0].im + m[1].re * m[1].re + m[1].im * m[1].im
                           + m[2].re * m[2].re + m[2].im * m[2].im);
    m[0] = n0 * m[0];
    m[1] = n0 * m[1];
    m[2] = n0 * m[2];
    cd psi = mul_c(m[3], m[0]) + mul_c(m[4], m[1]) + mul_c(m[5], m[2]);
    m[3] = m[3] - psi * m[0];
    m[4] = m[4] - psi * m[1];
    m[5] = m[5] - psi * m[2];
    double n1 = 1.0 / sqrt(m[3].re * m[3].re + m[3].im * m[3].im + m[4].re * m[4].re + m[4].im * m[4].im
                           + m[5].re * m[5].re + m[5].im * m[5].im);
    m[3] = n1 * m[3];
    m[4] = n1 * m[4];
    m[5] = n1 * m[5];
    m[6] = conj_cross(m[1], m[5], m[2], m[4]);
    m[7] = conj_cross(m[2], m[3], m[0], m[5]);
    m[8] = conj_cross(m[0], m[4], m[1], m[3]);
}

// ---------------------------------------------------------------------------
// Cayley-Hamilton exp(iQ) for traceless hermitian Q (Morningstar-Peardon),
// with the same branch structure and Taylor switch-over points as the
// reference's SU3::ExpConstants.
struct ExpC {
    double u, w, u2, w2, c0max;
    int signflip;
    cd exp_miu, exp_2iu, h0, h1, h2;
    double denom, cosw, xi0;
};

__device__ __forceinline__ double xi0_of(double w)
{
    if (fabs(w) <= 0.05) {
        double w2 = w * w;
        return 1.0 - (1.0 / 6.0) * w2 * (1.0 - (1.0 / 20.0) * w2 * (1.0 - (1.0 / 42.0) * w2));
    }
    return sin(w) / w;
}
__device__ __forceinline__ double xi1_of(double w)
{
    if (fabs(w) <= 0.115) {
        double w2 = w * w;
        return -(1.0 / 3.0) + (1.0 / 30.0) * w2 * (1.0 - (1.0 / 28.0) * w2 * (1.0 - (1.0 / 54.0) * w2));
    }
    return cos(w) / (w * w) - sin(w) / (w * w * w);
}

// From the invariants c0s = tr(Q^3)/3 = det Q and c1 = tr(Q^2)/2.
__device__ __forceinline__ void exp_constants_c(double c0s, double c1, ExpC& e)
{
    double c0 = fabs(c0s);
    const double c1_3 = c1 / 3.0;
    e.c0max = 2.0 * (c1_3 * sqrt(c1_3));   // 2 (c1/3)^(3/2)
    e.signflip = c0s < 0.0;
    double theta = acos(fmin(c0 / e.c0max, 1.0));
    double st, ct;
    sincos((1.0 / 3.0) * theta, &st, &ct);
    e.u = sqrt((1.0 / 3.0) * c1) * ct;
    e.w = sqrt(c1) * st;
    e.u2 = e.u * e.u;
    e.w2 = e.w * e.w;
    double su, cu;
    sincos(e.u, &su, &cu);
    e.exp_miu = cd{cu, -su};
    e.exp_2iu = conj(e.exp_miu * e.exp_miu);
    e.cosw = cos(e.w);
    e.xi0 = xi0_of(e.w);
    if (e.c0max < 2.2250738585072014e-308) {
        e.denom = 1.0;
        e.h0 = cd{1.0, 0.0};
        e.h1 = cd{0.0, 0.0};
        e.h2 = cd{0.0, 0.0};
        return;
    }
    const double u = e.u, u2 = e.u2, w2 = e.w2;
    const cd ixi0 = cd{0.0, e.xi0};
    e.denom = 1.0 / (9.0 * u2 - w2);
    cd h0 = (u2 - w2) * e.exp_2iu + e.exp_miu * (cd{8.0 * u2 * e.cosw, 0.0} + (2.0 * u) * ixi0 * (3.0 * u2 + w2));
    cd h1 = (2.0 * u) * e.exp_2iu - e.exp_miu * (cd{2.0 * u * e.cosw, 0.0} - ixi0 * (3.0 * u2 - w2));
    cd h2 = e.exp_2iu - e.exp_miu * (cd{e.cosw, 0.0} + (3.0 * u) * ixi0);
    if (e.signflip) {
        h0 = conj(h0);
        h1 = -conj(h1);
        h2 = conj(h2);
    }
    e.h0 = h0;
    e.h1 = h1;
    e.h2 = h2;
}

// exp(iQ) = f0 + f1 Q + f2 Q^2 by the power series reduced with Cayley-Hamilton: with
// Q^3 = c1 Q + c0 (c1 = tr Q^2 / 2, c0 = det Q) every power is Q^k = c0 G_{k-1} + G_{k+1} Q +
// G_k Q^2 where G_{k+1} = c1 G_{k-1} + c0 G_{k-2}, G_0 = G_1 = 0, G_2 = 1, so
//   f0 = 1 + c0 sum_k i^k/k! G_{k-1},  f1 = sum_k i^k/k! G_{k+1},  f2 = sum_k i^k/k! G_k:
// five FP64 instructions per term, no branches and no transcendental functions (the closed
// form above takes an arc cosine and three sine-cosine pairs).  The derivatives of G with
// respect to c1 and c0 are H_k and H_{k-1} with H_{k+1} = G_{k-1} + c1 H_{k-1} + c0 H_{k-2}
// (both have the generating function z^4 / (1 - c1 z^2 - c0 z^3)^2 up to a power of z), so
// the derivatives of f0, f1, f2 follow from one more sequence.
// The largest omitted terms of all eight coefficients are below 6e-18 with k <= 12 for
// c1 <= 0.02 (the Wilson flow's exponents) and 2e-18 with k <= 20 for c1 <= 1 (a stout step:
// c1 <= (6 rho)^2 3/2, 0.78 for rho = 0.12; the closed form loses digits to its denominator
// 9 u^2 - w^2 there).
constexpr double EXP_SERIES_SMALL = 0.02, EXP_SERIES_C1 = 1.0;
constexpr int EXP_TERMS_SMALL = 12, EXP_TERMS = 20;

// z += i^k t x.  k is a template argument all the way: with a run-time k in an unrolled loop
// the choice of re or im became a selected address, which kept z in scratch memory.
template <int K>
__device__ __forceinline__ void acc_ik(cd& z, double t, double x)
{
    constexpr int q = K & 3;
    if constexpr (q == 0) z.re = fma(t, x, z.re);
    if constexpr (q == 1) z.im = fma(t, x, z.im);
    if constexpr (q == 2) z.re = fma(-t, x, z.re);
    if constexpr (q == 3) z.im = fma(-t, x, z.im);
}
constexpr double inv_factorial(int k)
{
    double t = 1.0;
    for (int i = 2; i <= k; ++i) t /= (double)i;
    return t;
}
// the terms k .. K; gm, g, gp: G_{k-2}, G_{k-1}, G_k
template <int k, int K>
__device__ __forceinline__ void exp_terms(double c0, double c1, double gm, double g, double gp, cd& s0, cd& f1, cd& f2)
{
    constexpr double t = inv_factorial(k);
    const double next = k == 2 ? 0.0 : fma(c1, g, c0 * gm);
    if constexpr (k >= 3) acc_ik<k>(s0, t, g);
    acc_ik<k>(f2, t, gp);
    if constexpr (k >= 3) acc_ik<k>(f1, t, next);
    if constexpr (k < K) exp_terms<k + 1, K>(c0, c1, g, gp, next, s0, f1, f2);
}
struct ExpCoeffs {
    cd f0, f1, f2;
};
template <int K>
__device__ __forceinline__ ExpCoeffs exp_series(double c0, double c1)
{
    cd s0 = cd{0.0, 0.0}, f1 = cd{0.0, 1.0}, f2 = cd{0.0, 0.0};   // k = 1: G_2 = 1
    exp_terms<2, K>(c0, c1, 0.0, 0.0, 1.0, s0, f1, f2);
    return ExpCoeffs{cd{fma(c0, s0.re, 1.0), c0 * s0.im}, f1, f2};
}
// f0, f1, f2 and the derivatives b1j = df_j/dc1, b2j = df_j/dc0 (the b_ij of Morningstar-Peardon)
struct ExpDeriv {
    cd f0, f1, f2, b10, b11, b12, b20, b21, b22;
};
// sequences at term k: G_{k-2}, G_{k-1}, G_k and H_{k-3} .. H_k
struct ExpSeq {
    double gm, g, gp, hmm, hk1, hk, hp;
};
struct ExpSums {
    cd s0, f1, f2, h2, h1, h0, hm;
};
template <int k, int K>
__device__ __forceinline__ void exp_terms_deriv(double c0, double c1, const ExpSeq& q, ExpSums& s)
{
    constexpr double t = inv_factorial(k);
    const double gnext = k == 2 ? 0.0 : fma(c1, q.g, c0 * q.gm);
    const double hnext = k <= 2 ? 0.0 : (k == 3 ? 1.0 : fma(c1, q.hk, fma(c0, q.hk1, q.g)));   // H_{k+1}
    acc_ik<k>(s.f2, t, q.gp);
    if constexpr (k >= 3) {
        acc_ik<k>(s.s0, t, q.g);
        acc_ik<k>(s.f1, t, gnext);
        acc_ik<k>(s.h2, t, hnext);    // sum i^k/k! H_{k+1}
    }
    if constexpr (k >= 4) acc_ik<k>(s.h1, t, q.hp);
    if constexpr (k >= 5) acc_ik<k>(s.h0, t, q.hk);
    if constexpr (k >= 6) acc_ik<k>(s.hm, t, q.hk1);
    if constexpr (k < K)
        exp_terms_deriv<k + 1, K>(c0, c1, ExpSeq{q.g, q.gp, gnext, q.hk1, q.hk, q.hp, hnext}, s);
}
template <int K>
__device__ __forceinline__ void exp_series_deriv(double c0, double c1, ExpDeriv& d)
{
    ExpSums s{};
    s.f1 = cd{0.0, 1.0};
    exp_terms_deriv<2, K>(c0, c1, ExpSeq{0.0, 0.0, 1.0, 0.0, 0.0, 0.0, 0.0}, s);
    d.f0 = cd{fma(c0, s.s0.re, 1.0), c0 * s.s0.im};
    d.f1 = s.f1;
    d.f2 = s.f2;
    d.b10 = c0 * s.h0;
    d.b11 = s.h2;
    d.b12 = s.h1;
    d.b20 = cd{fma(c0, s.hm.re, s.s0.re), fma(c0, s.hm.im, s.s0.im)};
    d.b21 = s.h1;
    d.b22 = s.h0;
}
// By value: stores through references at the end of the three branches are merged into one
// store to a selected address, which put the coefficients in scratch memory.
__device__ __forceinline__ ExpCoeffs exp_coeffs(double c0, double c1)
{
    if (c1 <= EXP_SERIES_SMALL) return exp_series<EXP_TERMS_SMALL>(c0, c1);
    if (c1 <= EXP_SERIES_C1) return exp_series<EXP_TERMS>(c0, c1);
    ExpC e;
    exp_constants_c(c0, c1, e);
    return ExpCoeffs{e.denom * e.h0, e.denom * e.h1, e.denom * e.h2};
}

// exp(iQ)
__device__ __forceinline__ M3 su3_exp(const M3& Q)
{
    M3 Q2 = mul(Q, Q);
    const auto [f0, f1, f2] = exp_coeffs((1.0 / 3.0) * retr_mul(Q, Q2), 0.5 * (Q2.m[0].re + Q2.m[4].re + Q2.m[8].re));
    M3 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.m[i] = f1 * Q.m[i] + f2 * Q2.m[i];
    r.m[0] += f0;
    r.m[4] += f0;
    r.m[8] += f0;
    return r;
}

// exp(c * A) for traceless anti-hermitian A: exp(i * (-i c A))
__device__ __forceinline__ M3 exp_ah(const M3& A, double c)
{
    M3 Q;
#pragma unroll
    for (int i = 0; i < 9; ++i) Q.m[i] = cd{c * A.m[i].im, -c * A.m[i].re};   // -i c A
    return su3_exp(Q);
}

// ---------------------------------------------------------------------------
// Block reductions: a butterfly over the 64 lanes of each wavefront (cross-lane
// exchanges, no LDS round trip and no barrier per level), then the per-wave values
// in LDS combined in wave order by thread 0, which alone holds the result.  At each
// butterfly level lane i forms op(v_i, v_j) and lane j forms op(v_j, v_i); op is
// commutative, so all lanes of a wave agree and the result does not depend on the
// scheduling.  Every thread of the block must call it; the leading barrier lets a
// kernel call it more than once (thread 0 has read the previous call's LDS values).
struct OpAdd {
    template <typename T>
    __device__ __forceinline__ T operator()(T a, T b) const { return a + b; }
};
struct OpMax {
    __device__ __forceinline__ double operator()(double a, double b) const { return fmax(a, b); }
};
template <int BS, typename T, int N, typename Op>
__device__ __forceinline__ void block_reduce(T (&v)[N], Op op)
{
    static_assert(BS % 64 == 0 && BS <= 1024, "block of whole wavefronts");
    constexpr int NW = BS / 64;
    __shared__ T sh[N][NW];
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v[n] = op(v[n], __shfl_xor(v[n], o, 64));
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int n = 0; n < N; ++n) sh[n][threadIdx.x >> 6] = v[n];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int n = 0; n < N; ++n)
#pragma unroll
            for (int w = 1; w < NW; ++w) v[n] = op(v[n], sh[n][w]);
}
// sum of v over the block, written to *out by thread 0
template <int BS>
__device__ __forceinline__ void block_sum_to(double v, double* out)
{
    double a[1] = {v};
    block_reduce<BS>(a, OpAdd{});
    if (threadIdx.x == 0) *out = a[0];
}

// the sum of part[stride i], i < n, over one block of BS lanes, in a fixed order: lane i keeps
// eight running sums of the entries i + BS u (u < 8) of each group of 8 BS entries (eight
// loads in flight instead of one), the rest into the first, then a fixed pairing; the lanes
// are left to block_reduce
template <int BS>
__device__ __forceinline__ double partials_sum(const double* __restrict__ part, int n, int stride = 1)
{
    double a[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int i = threadIdx.x;
    for (; i + 7 * BS < n; i += 8 * BS)
#pragma unroll
        for (int u = 0; u < 8; ++u) a[u] += part[(size_t)stride * (i + u * BS)];
    for (; i < n; i += BS) a[0] += part[(size_t)stride * i];
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
}

// ---------------------------------------------------------------------------
// Philox4x32-10 counter RNG (Salmon et al., SC'11).  Counter layout:
//   key = seed, ctr = {site, stream<<24 | k<<4 | sub<<2 | mu, counter_lo, counter_hi}
enum : uint32_t { RNG_HEATBATH = 0, RNG_MOMENTUM = 1, RNG_HAAR = 2 };

__host__ __device__ __forceinline__ uint32_t mulhi32(uint32_t a, uint32_t b)
{
    return (uint32_t)(((uint64_t)a * b) >> 32);
}

__host__ __device__ __forceinline__ void philox10(uint32_t c[4], uint32_t k0, uint32_t k1)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        uint32_t hi0 = mulhi32(0xD2511F53u, c[0]);
        uint32_t lo0 = 0xD2511F53u * c[0];
        uint32_t hi1 = mulhi32(0xCD9E8D57u, c[2]);
        uint32_t lo1 = 0xCD9E8D57u * c[2];
        uint32_t n0 = hi1 ^ c[1] ^ k0;
        uint32_t n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
    }
}

__host__ __device__ __forceinline__ double u01(uint32_t a, uint32_t b)
{
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

__host__ __device__ __forceinline__ void draw2(uint64_t seed, uint32_t site, uint32_t stream, uint32_t k,
                                               uint32_t sub, uint32_t mu, uint64_t counter, double& u0, double& u1)
{
    uint32_t c[4] = {site, (stream << 24) | (k << 4) | (sub << 2) | mu, (uint32_t)counter, (uint32_t)(counter >> 32)};
    philox10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    u0 = u01(c[0], c[1]);
    u1 = u01(c[2], c[3]);
}

// Box-Muller pair from two uniforms
__device__ __forceinline__ void gauss2(double u0, double u1, double& g0, double& g1)
{
    double r = sqrt(-2.0 * log(1.0 - u0));
    double s, c;
    sincos(2.0 * 3.14159265358979323846 * u1, &s, &c);
    g0 = r * c;
    g1 = r * s;
}

// Division of 0 <= n < 2^31 by d as one high product and a shift: with sh = ceil(log2 d) - 1
// and m = ceil(2^(32 + sh) / d), m d - 2^(32 + sh) < d <= 2^(sh + 1), so n m / 2^(32 + sh)
// exceeds n / d by less than 1/d and the quotient is exact.  A division by a kernel argument
// is about twenty VALU instructions otherwise, also where the operands are uniform; the maps
// from a thread to its site take eight to ten of them (OR + HB updates of a 16^4 lattice 462 ->
// 448 us, four colours at 28 x 20 x 12 x 36 2025 -> 1968 us, the heatbath launch at 32^4 128 -> 124 us).
struct Div {
    uint32_t m;
    int sh;
    int d;
};
inline Div make_div(int d)
{
    Div v{0u, 0, d};
    if (d > 1) {
        int bits = 0;   // ceil(log2 d)
        while ((1ll << bits) < d) ++bits;
        v.sh = bits - 1;
        v.m = (uint32_t)(((1ull << (32 + v.sh)) + (uint64_t)d - 1) / (uint64_t)d);
    }
    return v;
}
__host__ __device__ __forceinline__ int div_by(int n, const Div& v)
{
    const int q = (int)((uint32_t)(((uint64_t)(uint32_t)n * v.m) >> 32) >> v.sh);
    return v.d == 1 ? n : q;
}
// n <- n / d, returns n % d
__host__ __device__ __forceinline__ int mod_div(int& n, const Div& v)
{
    const int q = div_by(n, v), r = n - q * v.d;
    n = q;
    return r;
}

// ---------------------------------------------------------------------------
// Lattice geometry.  Sites are lexicographic s = ((t*Nx+x)*Ny+y)*Nz+z; the parity
// of a site is (t+x+y+z)&1 and, because Nz is even, its checkerboard index is s>>1.
// Links live in a structure-of-arrays buffer of complex doubles:
//   U[((mu*2 + parity)*9 + c)*Vh + cbi(s)],  c = 3*row + col,  Vh = V/2,
// where cbi(s) is the checkerboard index s>>1 (plain order) or, in the four-colour
// sweep kernels, that index with each group of 16 ordered even ones first (below).
struct Geom {
    int L[4];       // Nt, Nx, Ny, Nz
    int st[4];      // lexicographic strides of t, x, y, z
    int V, Vh;
    Div dx, dy, dz; // division by Nx, Ny, Nz
};

// Storage slot of site s in its parity array.  Plain order: cb = s>>1.  Split order
// (translation units compiled with LT_SPLIT_CB = 1, the four-colour sweeps): within
// every aligned group of 16 checkerboard indices the 8 even ones come first, then the
// 8 odd ones, so a 256-byte group of one component becomes two 128-byte lines, one
// per cb parity (a last group of 8, when Vh is not a multiple of 16, keeps its
// order).  With Nz divisible by 4, cb & 1 is (z>>1) & 1, so a colour class of the
// four-colour schedule (every fourth z of a row) reads and writes whole lines instead
// of every other 16-byte slot.  The split order costs the two-colour and Jacobi
// kernels a few address instructions per link (measured at 32^4: RK3 flow stage
// +13 %, observables +22 %), so they keep the plain order.  Kernels address links
// only through this function: the order never changes a result.
#ifndef LT_SPLIT_CB
#define LT_SPLIT_CB 0
#endif
__device__ __forceinline__ int cbi(const Geom& g, int s)
{
    const int cb = s >> 1;
#if LT_SPLIT_CB
    const int p = (cb & ~15) | ((cb & 1) << 3) | ((cb >> 1) & 7);
    return cb < (g.Vh & ~15) ? p : cb;
#else
    return cb;
#endif
}

// Offset, in complex doubles, of slot 0 of storage position pos of array a (a =
// mu*2 + parity, or plane*2 + parity) in a buffer of nslot slots per entry, and the
// distance between consecutive slots of one entry: one array of Vh entries per slot.
// (Blocks of 8 positions holding their slots one after another were measured at 32^4:
// overrelaxation +3 %, heatbath -3 %, flow unchanged; not kept.)
__device__ __forceinline__ size_t slot_base(const Geom& g, int a, int nslot, int pos)
{
    return (size_t)a * (size_t)nslot * (size_t)g.Vh + (size_t)pos;
}
__device__ __forceinline__ size_t slot_stride(const Geom& g) { return (size_t)g.Vh; }

// v[i] for an index known only at run time, as four masked values: nested conditionals on
// kernel arguments become a tree of branches, which cuts every kernel that works with
// run-time directions into pieces that the compiler cannot schedule across.
__device__ __forceinline__ int pick4(const int v[4], int i)
{
    const int a = v[0], b = v[1], c = v[2], d = v[3];
    return (a & -(int)(i == 0)) | (b & -(int)(i == 1)) | (c & -(int)(i == 2)) | (d & -(int)(i == 3));
}

__device__ __forceinline__ void coords_of(const Geom& g, int s, int c[4])
{
    c[3] = mod_div(s, g.dz);
    c[2] = mod_div(s, g.dy);
    c[1] = mod_div(s, g.dx);
    c[0] = s;
}
// site index one step along +mu / -mu given the coordinate of that direction
__device__ __forceinline__ int up(const Geom& g, int s, int cmu, int mu)
{
    const int L = pick4(g.L, mu), st = pick4(g.st, mu);
    return (cmu + 1 < L) ? s + st : s - (L - 1) * st;
}
__device__ __forceinline__ int dn(const Geom& g, int s, int cmu, int mu)
{
    const int L = pick4(g.L, mu), st = pick4(g.st, mu);
    return (cmu > 0) ? s - st : s + (L - 1) * st;
}

// Element i of a buffer.  With LT_ADDR32 the byte offset is a 32-bit value added to
// the (wave-uniform) base pointer, which lets loads use the scalar-base +
// vector-offset form; buffers must then stay below 4 GiB.
#ifndef LT_ADDR32
#define LT_ADDR32 0
#endif
__device__ __forceinline__ const double2& elem(const double2* __restrict__ base, size_t i)
{
#if LT_ADDR32
    return *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(base) + (uint32_t)((uint32_t)i * 16u));
#else
    return base[i];
#endif
}
__device__ __forceinline__ double2& elem(double2* __restrict__ base, size_t i)
{
#if LT_ADDR32
    return *reinterpret_cast<double2*>(reinterpret_cast<char*>(base) + (uint32_t)((uint32_t)i * 16u));
#else
    return base[i];
#endif
}

__device__ __forceinline__ M3 ld(const double2* __restrict__ U, const Geom& g, int s, int mu, int par)
{
    const size_t o = slot_base(g, mu * 2 + par, 9, cbi(g, s));
    M3 r;
#pragma unroll
    for (int c = 0; c < 9; ++c) {
        double2 v = elem(U, o + (size_t)c * slot_stride(g));
        r.m[c] = cd{v.x, v.y};
    }
    return r;
}
__device__ __forceinline__ void st_link(double2* __restrict__ U, const Geom& g, int s, int mu, int par, const M3& a)
{
    const size_t o = slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 9; ++c) elem(U, o + (size_t)c * slot_stride(g)) = make_double2(a.m[c].re, a.m[c].im);
}
// su(3) algebra fields (anti-hermitian, traceless: the Wilson-flow Z) in 8 reals,
//   Z[((mu*2 + parity)*4 + c)*Vh + cb],  c: 0 = (Im a00, Im a11), 1 = a01, 2 = a02, 3 = a12;
// Re a_ii = 0, a_22 = -(a_00 + a_11) and a_ji = -conj(a_ij) are implied.
struct Alg8 {
    double d0, d1;
    cd a01, a02, a12;
};
__device__ __forceinline__ Alg8 to_alg8(const M3& a)
{
    return Alg8{a.m[0].im, a.m[4].im, a.m[1], a.m[2], a.m[5]};
}
__device__ __forceinline__ M3 from_alg8(const Alg8& z)
{
    M3 r;
    r.m[0] = cd{0.0, z.d0};
    r.m[4] = cd{0.0, z.d1};
    r.m[8] = cd{0.0, -(z.d0 + z.d1)};
    r.m[1] = z.a01;
    r.m[2] = z.a02;
    r.m[5] = z.a12;
    r.m[3] = cd{-z.a01.re, z.a01.im};
    r.m[6] = cd{-z.a02.re, z.a02.im};
    r.m[7] = cd{-z.a12.re, z.a12.im};
    return r;
}
__device__ __forceinline__ Alg8 scale(double a, const Alg8& x)
{
    return Alg8{a * x.d0, a * x.d1, a * x.a01, a * x.a02, a * x.a12};
}
// a * x + b * y
__device__ __forceinline__ Alg8 axpby(double a, const Alg8& x, double b, const Alg8& y)
{
    return Alg8{a * x.d0 + b * y.d0, a * x.d1 + b * y.d1, a * x.a01 + b * y.a01, a * x.a02 + b * y.a02,
                a * x.a12 + b * y.a12};
}
__device__ __forceinline__ Alg8 ld_alg8(const double2* __restrict__ Z, const Geom& g, int s, int mu, int par)
{
    const double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    const double2 v0 = p[0], v1 = p[slot_stride(g)], v2 = p[(size_t)2 * slot_stride(g)], v3 = p[(size_t)3 * slot_stride(g)];
    return Alg8{v0.x, v0.y, cd{v1.x, v1.y}, cd{v2.x, v2.y}, cd{v3.x, v3.y}};
}
__device__ __forceinline__ void st_alg8(double2* __restrict__ Z, const Geom& g, int s, int mu, int par, const Alg8& z)
{
    double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    p[0] = make_double2(z.d0, z.d1);
    p[slot_stride(g)] = make_double2(z.a01.re, z.a01.im);
    p[(size_t)2 * slot_stride(g)] = make_double2(z.a02.re, z.a02.im);
    p[(size_t)3 * slot_stride(g)] = make_double2(z.a12.re, z.a12.im);
}

// Streaming (non-temporal) accesses for data touched once per launch, so that it
// does not displace the L2-resident neighbourhood of the link reads.
typedef double lt_d2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double2 ld_stream(const double2* p)
{
    const lt_d2v v = __builtin_nontemporal_load(reinterpret_cast<const lt_d2v*>(p));
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void st_stream(double2* p, double2 v)
{
    const lt_d2v w = {v.x, v.y};
    __builtin_nontemporal_store(w, reinterpret_cast<lt_d2v*>(p));
}
__device__ __forceinline__ Alg8 ld_alg8_stream(const double2* __restrict__ Z, const Geom& g, int s, int mu, int par)
{
    const double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    const double2 v0 = ld_stream(p), v1 = ld_stream(p + slot_stride(g)), v2 = ld_stream(p + (size_t)2 * slot_stride(g)),
                  v3 = ld_stream(p + (size_t)3 * slot_stride(g));
    return Alg8{v0.x, v0.y, cd{v1.x, v1.y}, cd{v2.x, v2.y}, cd{v3.x, v3.y}};
}
__device__ __forceinline__ void st_alg8_stream(double2* __restrict__ Z, const Geom& g, int s, int mu, int par,
                                               const Alg8& z)
{
    double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    st_stream(p, make_double2(z.d0, z.d1));
    st_stream(p + slot_stride(g), make_double2(z.a01.re, z.a01.im));
    st_stream(p + (size_t)2 * slot_stride(g), make_double2(z.a02.re, z.a02.im));
    st_stream(p + (size_t)3 * slot_stride(g), make_double2(z.a12.re, z.a12.im));
}

// Traceless hermitian fields (the stout exponents Q of the CV tape, the stout-force
// Lambda) in 8 reals, slots as above:
//   c: 0 = (Re q00, Re q11), 1 = q01, 2 = q02, 3 = q12;
// Im q_ii = 0, q_22 = -(q_00 + q_11) and q_ji = conj(q_ij) are implied.
__device__ __forceinline__ void st_her8(double2* __restrict__ Z, const Geom& g, int s, int mu, int par, const M3& q)
{
    double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    p[0] = make_double2(q.m[0].re, q.m[4].re);
    p[slot_stride(g)] = make_double2(q.m[1].re, q.m[1].im);
    p[(size_t)2 * slot_stride(g)] = make_double2(q.m[2].re, q.m[2].im);
    p[(size_t)3 * slot_stride(g)] = make_double2(q.m[5].re, q.m[5].im);
}
// Hermitian or anti-hermitian 3x3 matrices in 9 reals: the diagonal (d, or i d where AH) and
// the upper triangle; the lower triangle is conj (-conj where AH) of the upper one.
struct Tri {
    double d0, d1, d2;
    cd r01, r02, r12;
};
// Q^2 of a hermitian Q from its six independent entries
__device__ __forceinline__ Tri her_square(const Tri& q)
{
    const double n01 = q.r01.re * q.r01.re + q.r01.im * q.r01.im, n02 = q.r02.re * q.r02.re + q.r02.im * q.r02.im,
                 n12 = q.r12.re * q.r12.re + q.r12.im * q.r12.im;
    return Tri{fma(q.d0, q.d0, n01 + n02),
               fma(q.d1, q.d1, n01 + n12),
               fma(q.d2, q.d2, n02 + n12),
               (q.d0 + q.d1) * q.r01 + mul_c(q.r02, q.r12),
               (q.d0 + q.d2) * q.r02 + q.r01 * q.r12,
               (q.d1 + q.d2) * q.r12 + cmul(q.r01, q.r02)};
}
__device__ __forceinline__ double her_det(const Tri& q)
{
    const cd t = q.r01 * q.r12;
    const double n01 = q.r01.re * q.r01.re + q.r01.im * q.r01.im, n02 = q.r02.re * q.r02.re + q.r02.im * q.r02.im,
                 n12 = q.r12.re * q.r12.re + q.r12.im * q.r12.im;
    return q.d0 * q.d1 * q.d2 - q.d0 * n12 - q.d1 * n02 - q.d2 * n01 + 2.0 * (t.re * q.r02.re + t.im * q.r02.im);
}
// f0 + f1 Q + f2 Q^2, s = Q^2
__device__ __forceinline__ M3 her_poly(cd f0, cd f1, cd f2, const Tri& q, const Tri& s)
{
    M3 r;
    r.m[0] = f0 + q.d0 * f1 + s.d0 * f2;
    r.m[4] = f0 + q.d1 * f1 + s.d1 * f2;
    r.m[8] = f0 + q.d2 * f1 + s.d2 * f2;
    r.m[1] = f1 * q.r01 + f2 * s.r01;
    r.m[2] = f1 * q.r02 + f2 * s.r02;
    r.m[5] = f1 * q.r12 + f2 * s.r12;
    r.m[3] = f1 * conj(q.r01) + f2 * conj(s.r01);
    r.m[6] = f1 * conj(q.r02) + f2 * conj(s.r02);
    r.m[7] = f1 * conj(q.r12) + f2 * conj(s.r12);
    return r;
}
// exp(iQ) for Q hermitian traceless: Q^2 from its six independent entries, c0 = det Q and
// c1 = tr(Q^2)/2 from Q's entries
__device__ __forceinline__ M3 exp_her(const Tri& q)
{
    const Tri s = her_square(q);
    const auto [f0, f1, f2] = exp_coeffs(her_det(q), 0.5 * (s.d0 + s.d1 + s.d2));
    return her_poly(f0, f1, f2, q, s);
}
// exp(c Z) for Z anti-hermitian traceless in the 8-real form (the flow's Z): exp(iQ) with
// Q = -i c Z hermitian traceless
__device__ __forceinline__ M3 exp_alg8(const Alg8& z, double c)
{
    const double q0 = c * z.d0, q1 = c * z.d1;
    return exp_her(Tri{q0, q1, -(q0 + q1), cd{c * z.a01.im, -c * z.a01.re}, cd{c * z.a02.im, -c * z.a02.re},
                       cd{c * z.a12.im, -c * z.a12.re}});
}
__device__ __forceinline__ Tri ld_her8_tri(const double2* __restrict__ Z, const Geom& g, int s, int mu, int par)
{
    const double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
    const double2 v0 = p[0], v1 = p[slot_stride(g)], v2 = p[(size_t)2 * slot_stride(g)], v3 = p[(size_t)3 * slot_stride(g)];
    return Tri{v0.x, v0.y, -(v0.x + v0.y), cd{v1.x, v1.y}, cd{v2.x, v2.y}, cd{v3.x, v3.y}};
}
__device__ __forceinline__ Tri operator-(const Tri& a, const Tri& b)
{
    return Tri{a.d0 - b.d0, a.d1 - b.d1, a.d2 - b.d2, a.r01 - b.r01, a.r02 - b.r02, a.r12 - b.r12};
}
// c += SG a d (i a d where AH), SG = +-1
template <bool AH, int SG>
__device__ __forceinline__ void diag_acc(cd& c, cd a, double d)
{
    if (AH) {
        c.re = fma(SG > 0 ? -a.im : a.im, d, c.re);
        c.im = fma(SG > 0 ? a.re : -a.re, d, c.im);
    } else {
        c.re = fma(SG > 0 ? a.re : -a.re, d, c.re);
        c.im = fma(SG > 0 ? a.im : -a.im, d, c.im);
    }
}
// c += SG a b
template <int SG>
__device__ __forceinline__ void cmul_acc(cd& c, cd a, cd b)
{
    const double s = SG > 0 ? 1.0 : -1.0;
    c.re = fma(s * a.re, b.re, c.re);
    c.re = fma(-s * a.im, b.im, c.re);
    c.im = fma(s * a.re, b.im, c.im);
    c.im = fma(s * a.im, b.re, c.im);
}
// C += SG A R and C += SG R A for R hermitian (AH: anti-hermitian): 10 FP64 instructions per
// complex entry instead of 12, the zero parts of the diagonal left out
template <bool AH, int SG>
__device__ __forceinline__ void mul_tri_acc(M3& C, const M3& A, const Tri& R)
{
    constexpr int LO = AH ? -SG : SG;   // sign of the conjugated lower triangle
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const cd x = A.m[3 * i], y = A.m[3 * i + 1], z = A.m[3 * i + 2];
        diag_acc<AH, SG>(C.m[3 * i], x, R.d0);
        cmul_acc<LO>(C.m[3 * i], y, conj(R.r01));
        cmul_acc<LO>(C.m[3 * i], z, conj(R.r02));
        cmul_acc<SG>(C.m[3 * i + 1], x, R.r01);
        diag_acc<AH, SG>(C.m[3 * i + 1], y, R.d1);
        cmul_acc<LO>(C.m[3 * i + 1], z, conj(R.r12));
        cmul_acc<SG>(C.m[3 * i + 2], x, R.r02);
        cmul_acc<SG>(C.m[3 * i + 2], y, R.r12);
        diag_acc<AH, SG>(C.m[3 * i + 2], z, R.d2);
    }
}
template <bool AH, int SG>
__device__ __forceinline__ void tri_mul_acc(M3& C, const Tri& R, const M3& A)
{
    constexpr int LO = AH ? -SG : SG;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const cd x = A.m[j], y = A.m[3 + j], z = A.m[6 + j];
        diag_acc<AH, SG>(C.m[j], x, R.d0);
        cmul_acc<SG>(C.m[j], R.r01, y);
        cmul_acc<SG>(C.m[j], R.r02, z);
        cmul_acc<LO>(C.m[3 + j], conj(R.r01), x);
        diag_acc<AH, SG>(C.m[3 + j], y, R.d1);
        cmul_acc<SG>(C.m[3 + j], R.r12, z);
        cmul_acc<LO>(C.m[6 + j], conj(R.r02), x);
        cmul_acc<LO>(C.m[6 + j], conj(R.r12), y);
        diag_acc<AH, SG>(C.m[6 + j], z, R.d2);
    }
}

// One 8-real algebra or hermitian entry as loaded
struct Raw4 {
    double2 v[4];
};
__device__ __forceinline__ void ld_raw4(const double2* __restrict__ Z, const Geom& g, int s, int mu, int par, Raw4& r)
{
    const double2* p = Z + slot_base(g, mu * 2 + par, 4, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 4; ++c) r.v[c] = p[(size_t)c * slot_stride(g)];
}
__device__ __forceinline__ Tri her_of(const Raw4& r)
{
    return Tri{r.v[0].x, r.v[0].y, -(r.v[0].x + r.v[0].y), cd{r.v[1].x, r.v[1].y}, cd{r.v[2].x, r.v[2].y},
               cd{r.v[3].x, r.v[3].y}};
}
__device__ __forceinline__ Tri ah_tri(const M3& a) { return Tri{a.m[0].im, a.m[4].im, a.m[8].im, a.m[1], a.m[2], a.m[5]}; }
// A + R, R anti-hermitian
__device__ __forceinline__ M3 add_ah(M3 a, const Tri& r)
{
    a.m[0].im += r.d0;
    a.m[4].im += r.d1;
    a.m[8].im += r.d2;
    a.m[1] += r.r01;
    a.m[2] += r.r02;
    a.m[5] += r.r12;
    a.m[3] += cd{-r.r01.re, r.r01.im};
    a.m[6] += cd{-r.r02.re, r.r02.im};
    a.m[7] += cd{-r.r12.re, r.r12.im};
    return a;
}
// A B where the product is known to be anti-hermitian and traceless
__device__ __forceinline__ Tri mul_ah(const M3& A, const M3& B)
{
    auto entry = [&](int i, int j) {
        cd z = A.m[3 * i] * B.m[j];
        cmul_acc<1>(z, A.m[3 * i + 1], B.m[3 + j]);
        cmul_acc<1>(z, A.m[3 * i + 2], B.m[6 + j]);
        return z;
    };
    auto diag = [&](int i) {
        double d = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k) d = fma(A.m[3 * i + k].re, B.m[3 * k + i].im, fma(A.m[3 * i + k].im, B.m[3 * k + i].re, d));
        return d;
    };
    const double d0 = diag(0), d1 = diag(1);
    return Tri{d0, d1, -(d0 + d1), entry(0, 1), entry(0, 2), entry(1, 2)};
}
// An anti-hermitian traceless field in 8 reals in the first four of the nine slots of a link
// field's entry
__device__ __forceinline__ void ld_ah8(const double2* __restrict__ S, const Geom& g, int s, int mu, int par, Raw4& r)
{
    const double2* p = S + slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 4; ++c) r.v[c] = p[(size_t)c * slot_stride(g)];
}
__device__ __forceinline__ void st_ah8(double2* __restrict__ S, const Geom& g, int s, int mu, int par, const Tri& y)
{
    double2* p = S + slot_base(g, mu * 2 + par, 9, cbi(g, s));
    p[0] = make_double2(y.d0, y.d1);
    p[slot_stride(g)] = make_double2(y.r01.re, y.r01.im);
    p[(size_t)2 * slot_stride(g)] = make_double2(y.r02.re, y.r02.im);
    p[(size_t)3 * slot_stride(g)] = make_double2(y.r12.re, y.r12.im);
}

// complex-double offset of a replica's 8-real field given its link-field offset
__host__ __device__ constexpr long long alg_offset(long long link_off) { return link_off / 72 * 32; }

// SU(3) links are stored as rows 0 and 1 only: every update ends with the
// Gram-Schmidt step whose last row is conj(row0 x row1), so row 2 is rebuilt on
// load with exactly that formula and never travels through memory.
__device__ __forceinline__ void third_row(M3& a)
{
    cd* m = a.m;
    m[6] = conj_cross(m[1], m[5], m[2], m[4]);
    m[7] = conj_cross(m[2], m[3], m[0], m[5]);
    m[8] = conj_cross(m[0], m[4], m[1], m[3]);
}
// acc + conj(x * y - z * w)
__device__ __forceinline__ cd conj_cross_acc(cd acc, cd x, cd y, cd z, cd w)
{
    double re = fma(z.im, w.im, acc.re);
    re = fma(-z.re, w.re, re);
    re = fma(-x.im, y.im, re);
    re = fma(x.re, y.re, re);
    double im = fma(z.im, w.re, acc.im);
    im = fma(z.re, w.im, im);
    im = fma(-x.im, y.re, im);
    im = fma(-x.re, y.im, im);
    return cd{re, im};
}
// acc += t for an SU(3) matrix t given by rows 0 and 1 (row 2 = conj(row0 x row1))
__device__ __forceinline__ void acc_su3_r01(M3& acc, const M3& t)
{
    const cd* m = t.m;
#pragma unroll
    for (int i = 0; i < 6; ++i) acc.m[i] += m[i];
    acc.m[6] = conj_cross_acc(acc.m[6], m[1], m[5], m[2], m[4]);
    acc.m[7] = conj_cross_acc(acc.m[7], m[2], m[3], m[0], m[5]);
    acc.m[8] = conj_cross_acc(acc.m[8], m[0], m[4], m[1], m[3]);
}
__device__ __forceinline__ M3 ldu(const double2* __restrict__ U, const Geom& g, int s, int mu, int par)
{
    const size_t o = slot_base(g, mu * 2 + par, 9, cbi(g, s));
    M3 r;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        double2 v = elem(U, o + (size_t)c * slot_stride(g));
        r.m[c] = cd{v.x, v.y};
    }
    third_row(r);
    return r;
}
// rows 0 and 1 of an SU(3) link; row 2 is left zero (callers never read it)
__device__ __forceinline__ M3 ldu2(const double2* __restrict__ U, const Geom& g, int s, int mu, int par)
{
    const size_t o = slot_base(g, mu * 2 + par, 9, cbi(g, s));
    M3 r;
#pragma unroll
    for (int c = 0; c < 6; ++c) {
        double2 v = elem(U, o + (size_t)c * slot_stride(g));
        r.m[c] = cd{v.x, v.y};
    }
    r.m[6] = r.m[7] = r.m[8] = cd{0.0, 0.0};
    return r;
}
__device__ __forceinline__ void stu(double2* __restrict__ U, const Geom& g, int s, int mu, int par, const M3& a)
{
    const size_t o = slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 6; ++c) elem(U, o + (size_t)c * slot_stride(g)) = make_double2(a.m[c].re, a.m[c].im);
}

__device__ __forceinline__ void stu_stream(double2* __restrict__ U, const Geom& g, int s, int mu, int par, const M3& a)
{
    double2* p = U + slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 6; ++c) st_stream(p + (size_t)c * slot_stride(g), make_double2(a.m[c].re, a.m[c].im));
}

// Clover planes R_munu = C_munu - C_munu^+ (mu < nu) are stored anti-hermitian in
// 9 reals, R_SLOTS complex slots per (plane, parity): 12 * R_SLOTS * Vh complex
// doubles per lattice; a replica at link offset off (72 * Vh units) has its
// planes at clover_offset(off).
constexpr int R_SLOTS = 5;
__host__ __device__ constexpr long long clover_offset(long long link_off) { return link_off / 72 * (12 * R_SLOTS); }

__device__ __forceinline__ int parity_of(const int c[4]) { return (c[0] + c[1] + c[2] + c[3]) & 1; }

// Thread -> site map of the per-parity link kernels.  Blocks cover 4D tiles of
// (t, x, y, zc) with zc = z/2 the checkerboard coordinate, z fastest inside a tile.
// The t tiles are split into chunks of tc consecutive tiles; tiles are ordered
// (t within the chunk) fastest, then z, y, x, chunk.  With tc = N[0]/8 each XCD's
// contiguous block range is one t-slab and the t-neighbours of a tile run a few
// blocks apart, inside the set of blocks resident in that XCD's L2.  The block
// index is first spread over XCDs.
//
// Linear maps (lin = 1) cover instead nthreads consecutive checkerboard sites of the
// parity per block (T = (1, 1, 1, nthreads), N = (blocks, 1, 1, 1)).  They serve extents
// whose z/2 has few factors of two (12^4, 20^4, 24^4: a dividing power-of-two box holds 2
// or 4 sites of a row, so a wavefront reads 32- or 64-byte pieces of 32 rows), where
// consecutive sites read whole rows and the t-slab of each XCD stays contiguous.
struct LinkMap {
    int T[4];     // tile extent in t, x, y, zc
    int N[4];     // number of tiles in t, x, y, zc
    int nthreads; // T[0]*T[1]*T[2]*T[3] == blockDim.x
    int tc;       // t tiles per chunk (divides N[0])
    int yc;       // y tiles per chunk (divides N[2]) of the Jacobi kernels (flow, stout, MetaD)
    int lin;      // linear map: block b covers checkerboard sites [b * nthreads, (b + 1) * nthreads)
    int xr;       // spread the block index over the XCDs (xcd_block)
    // divisions of map_site_b, from the numbers above (finish_map)
    Div dtx, dty, dtz, dtc, dnz, dyc, dnx, dny;
};
// to be called after any change of T, N, tc or yc
inline void finish_map(LinkMap& m)
{
    m.dtx = make_div(m.T[1]);
    m.dty = make_div(m.T[2]);
    m.dtz = make_div(m.T[3]);
    m.dtc = make_div(m.tc);
    m.dnz = make_div(m.N[3]);
    m.dyc = make_div(m.yc);
    m.dnx = make_div(m.N[1]);
    m.dny = make_div(m.N[2] / m.yc);
}

// Blocks of the split colour launches (64 links each): every timeslice of the class, nt
// links, is covered by its own blocks, the last one partly; the tc timeslices of a chunk are
// walked fastest, so that the t-neighbours of a block run in the same XCD at about the same
// time (24^4, Luescher-Weisz staple: 97 -> 85 us per overrelaxation launch with tc = 3; 20^4,
// four colours, Wilson staple: 25 -> 20 us with tc = 2).
constexpr int SPLIT_LINKS = 64;
struct SplitMap {
    int nt;
    Div dtc, dper;   // by tc, and by the blocks of a chunk
};

// Block index of a link kernel in its map's order: spread over the XCDs when m.xr is set.
__device__ __forceinline__ int link_block(const LinkMap& m, int b, int nb) { return m.xr ? xcd_block(b, nb) : b; }

// tile order, fastest first: t within its chunk, z, y within its chunk, x, y chunk, t chunk
__device__ __forceinline__ int site_of_cb(const Geom& g, int cb, int par, int c[4]);
__device__ __forceinline__ bool map_site_b(const Geom& g, const LinkMap& m, int b, int par, int c[4], int& s)
{
    int tid = threadIdx.x;
    if (m.lin) {
        const int cb = b * m.nthreads + tid;
        if (tid >= m.nthreads || cb >= g.Vh) return false;
        s = site_of_cb(g, cb, par, c);
        return true;
    }
    const int bt_lo = mod_div(b, m.dtc);
    const int bz = mod_div(b, m.dnz);
    const int by_lo = mod_div(b, m.dyc);
    const int bx = mod_div(b, m.dnx);
    const int by = mod_div(b, m.dny) * m.yc + by_lo;
    const int bt = b * m.tc + bt_lo;
    if (bt >= m.N[0] || tid >= m.nthreads) return false;
    const int dz = mod_div(tid, m.dtz);
    const int dy = mod_div(tid, m.dty);
    const int dx = mod_div(tid, m.dtx);
    const int dt = tid;
    c[0] = bt * m.T[0] + dt;
    c[1] = bx * m.T[1] + dx;
    c[2] = by * m.T[2] + dy;
    const int zc = bz * m.T[3] + dz;
    const int flip = (c[0] + c[1] + c[2] + par) & 1;
    c[3] = 2 * zc + flip;
    s = ((c[0] * g.L[1] + c[1]) * g.L[2] + c[2]) * g.L[3] + c[3];
    return true;
}

__device__ __forceinline__ bool map_site(const Geom& g, const LinkMap& m, int par, int c[4], int& s)
{
    return map_site_b(g, m, link_block(m, blockIdx.x, gridDim.x), par, c, s);
}

// Jacobi kernels over all links: the 8 (mu, parity) classes of one tile are
// consecutive blocks of the same XCD, so the staples of all directions at a tile
// are built from one L2-resident neighbourhood.  Grid: 8 * tiles blocks.
__device__ __forceinline__ bool map_link_b(const Geom& g, const LinkMap& m, int b, int& mu, int& par, int c[4], int& s)
{
    int mp = b & 7;
    mu = mp >> 1;
    par = mp & 1;
    return map_site_b(g, m, b >> 3, par, c, s);
}
__device__ __forceinline__ bool map_link_all(const Geom& g, const LinkMap& m, int& mu, int& par, int c[4], int& s)
{
    return map_link_b(g, m, link_block(m, blockIdx.x, gridDim.x), mu, par, c, s);
}

// Site of the cb-th entry of a parity: s = 2*cb or 2*cb+1 with the right parity.
__device__ __forceinline__ int site_of_cb(const Geom& g, int cb, int par, int c[4])
{
    int s = 2 * cb;
    coords_of(g, s, c);
    int flip = (c[0] + c[1] + c[2] + par) & 1;   // z of s is even
    c[3] += flip;
    return s + flip;
}

// Sites of the site kernels: 64 consecutive indices i are 32 checkerboard positions, first
// their parity-0 sites, then their parity-1 sites, so that each half wavefront reads 512
// consecutive bytes per component.  Walking sites in lexicographic order instead alternates
// the parity arrays from lane to lane, and the L1 then takes twice the accesses per load (32
// instead of 16; four times where the direction alternates too).  half_cb may pass the last
// position where their number is not a multiple of 32.
__device__ __forceinline__ int half_cb(int i) { return ((i >> 6) << 5) | (i & 31); }
__device__ __forceinline__ int half_par(int i) { return (i >> 5) & 1; }

// Staple of link (s, mu): sum over nu != mu (ascending) of
//   U_nu(x) U_mu(x+nu) U_nu(x+mu)^+ + U_nu(x-nu)^+ U_mu(x-nu) U_nu(x-nu+mu)
// Every partial product of links is in SU(3), so only its rows 0 and 1 are
// multiplied out and row 2 follows as conj(row0 x row1) (24 instead of 36 FP64
// instructions); the leading link of each product is read as rows 0 and 1 only.
// Upper term: (a b) c^+ with rows 0, 1 of both products; lower term:
// d^+ (e f) with rows 0, 1 of e f.  About 20 % fewer FP64 instructions than
// three full products per term.
__device__ __forceinline__ M3 staple(const double2* __restrict__ U, const Geom& g, int s, const int c[4], int mu)
{
    const int par = (c[0] + c[1] + c[2] + c[3]) & 1;
    const int s_mu = up(g, s, pick4(c, mu), mu);
    M3 st;
#pragma unroll
    for (int nu = 0, k = 0; nu < 4; ++nu) {
        if (nu == mu) continue;
        const int cnu = c[nu];
        const int s_nu = up(g, s, cnu, nu);
        const int s_nd = dn(g, s, cnu, nu);
        const int s_nd_mu = up(g, s_nd, pick4(c, mu), mu);
        {
            const M3 ab = mul_r01(ldu2(U, g, s, nu, par), ldu(U, g, s_nu, mu, par ^ 1));
            const M3 t = mul_nd_r01(ab, ldu(U, g, s_mu, nu, par ^ 1));
            if (k == 0) {
                st = t;
                third_row(st);
            } else {
                acc_su3_r01(st, t);
            }
        }
        {
            M3 ef = mul_r01(ldu2(U, g, s_nd, mu, par ^ 1), ldu(U, g, s_nd_mu, nu, par));
            third_row(ef);
            mul_dn_acc(st, ldu(U, g, s_nd, nu, par ^ 1), ef);
        }
        ++k;
    }
    return st;
}

// Rows 0 and 1 of one link as loaded (six complex entries).
struct Raw6 {
    double2 v[6];
};
__device__ __forceinline__ void ld_raw(const double2* __restrict__ U, const Geom& g, int s, int mu, int par, Raw6& r)
{
    const double2* p = U + slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int c = 0; c < 6; ++c) r.v[c] = p[(size_t)c * slot_stride(g)];
}
__device__ __forceinline__ M3 rows01(const Raw6& r)
{
    M3 a;
#pragma unroll
    for (int c = 0; c < 6; ++c) a.m[c] = cd{r.v[c].x, r.v[c].y};
    a.m[6] = a.m[7] = a.m[8] = cd{0.0, 0.0};
    return a;
}
__device__ __forceinline__ M3 su3_of(const Raw6& r)
{
    M3 a = rows01(r);
    third_row(a);
    return a;
}
// The staple of staple() as six terms (upper and lower for each nu != mu, nu
// ascending, the same products and summation order), software-pipelined: the
// three links of term j+1 are loaded before term j is multiplied out, with
// scheduling barriers so the compiler keeps that order instead of hoisting all
// 19 link loads (which spills).  The own link is loaded with the last term.
__device__ __forceinline__ M3 staple_pipelined(const double2* __restrict__ U, const Geom& g, int s, const int c[4],
                                               int mu, int par, Raw6& own)
{
    const int q = par ^ 1;
    const int s_mu = up(g, s, pick4(c, mu), mu);
    int s_nu[3], s_nd[3], s_ndmu[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int nu = k + (k >= mu);
        const int cnu = pick4(c, nu), L = pick4(g.L, nu), st = pick4(g.st, nu);
        s_nu[k] = (cnu + 1 < L) ? s + st : s - (L - 1) * st;
        s_nd[k] = (cnu > 0) ? s - st : s + (L - 1) * st;
        s_ndmu[k] = up(g, s_nd[k], pick4(c, mu), mu);
    }
    // term j = 2k: a = U_nu(x) [rows 0, 1], b = U_mu(x+nu), cc = U_nu(x+mu):  (a b) cc^+
    // term j = 2k+1: a = U_mu(x-nu) [rows 0, 1], b = U_nu(x-nu+mu), cc = U_nu(x-nu):  cc^+ (a b)
    auto load = [&](int j, Raw6& a, Raw6& b, Raw6& cc) {
        const int k = j >> 1, nu = k + (k >= mu);
        if ((j & 1) == 0) {
            ld_raw(U, g, s, nu, par, a);
            ld_raw(U, g, s_nu[k], mu, q, b);
            ld_raw(U, g, s_mu, nu, q, cc);
        } else {
            ld_raw(U, g, s_nd[k], mu, q, a);
            ld_raw(U, g, s_ndmu[k], nu, par, b);
            ld_raw(U, g, s_nd[k], nu, q, cc);
        }
    };
    Raw6 A[2], B[2], C[2];
    load(0, A[0], B[0], C[0]);
    M3 st;
#pragma unroll
    for (int j = 0; j < 6; ++j) {
        if (j < 5) load(j + 1, A[(j + 1) & 1], B[(j + 1) & 1], C[(j + 1) & 1]);
        if (j == 4) ld_raw(U, g, s, mu, par, own);
        __builtin_amdgcn_sched_barrier(0);
        const int i = j & 1;
        if ((j & 1) == 0) {
            const M3 t = mul_nd_r01(mul_r01(rows01(A[i]), su3_of(B[i])), su3_of(C[i]));
            if (j == 0) {
                st = t;
                third_row(st);
            } else {
                acc_su3_r01(st, t);
            }
        } else {
            M3 ef = mul_r01(rows01(A[i]), su3_of(B[i]));
            third_row(ef);
            mul_dn_acc(st, su3_of(C[i]), ef);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    return st;
}

// site x + a e_mu + b e_nu (|a|, |b| <= 2, mu != nu) of site s with coordinates c
__device__ __forceinline__ int wrap_add(int v, int a, int L)
{
    v += a;
    return v < 0 ? v + L : (v >= L ? v - L : v);
}
__device__ __forceinline__ int shift2(const Geom& g, int s, const int c[4], int mu, int a, int nu, int b)
{
    const int cm = pick4(c, mu), cn = pick4(c, nu);
    return s + (wrap_add(cm, a, pick4(g.L, mu)) - cm) * pick4(g.st, mu) +
           (wrap_add(cn, b, pick4(g.L, nu)) - cn) * pick4(g.st, nu);
}

// Parking: a matrix waits in LDS (9 entries at park[e * n], one slot per lane) while
// other work runs, so it holds no registers meanwhile; the empty asm statements with
// memory clobbers keep the compiler from carrying it in registers anyway.
__device__ __forceinline__ void park_store(double2* park, int n, const M3& a)
{
#pragma unroll
    for (int e = 0; e < 9; ++e) park[e * n] = make_double2(a.m[e].re, a.m[e].im);
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ M3 park_load(const double2* park, int n)
{
    asm volatile("" ::: "memory");
    M3 a;
#pragma unroll
    for (int e = 0; e < 9; ++e) a.m[e] = cd{park[e * n].x, park[e * n].y};
    return a;
}

// r += leaf - leaf^+ for an SU(3) leaf given by rows 0 and 1 (row 2 = conj(row0 x row1))
__device__ __forceinline__ void acc_leaf(Tri& r, M3& t)
{
    third_row(t);
    const cd* m = t.m;
    r.d0 += m[0].im + m[0].im;
    r.d1 += m[4].im + m[4].im;
    r.d2 += m[8].im + m[8].im;
    r.r01 += m[1] - conj(m[3]);
    r.r02 += m[2] - conj(m[6]);
    r.r12 += m[5] - conj(m[7]);
}
// R = C - C^+ (anti-hermitian, 9 reals) of the clover term C of plane (mu, nu) at site s: the
// four leaves in the orientation of the reference's CalculateClover<1,1>; retr: Re tr of leaf
// I, the plaquette.  Every leaf is a product of four links, an SU(3) matrix of which rows 0
// and 1 are multiplied out; only the nine reals of R are summed.  Each link is loaded two
// products ahead of the one that takes it (U_mu(x) a second time for leaf IV); the scheduling
// barriers keep the compiler from hoisting all loads (which spills).
__device__ __forceinline__ Tri clover_ah(const double2* __restrict__ U, const Geom& g, int s, const int c[4], int par,
                                         int mu, int nu, double& retr)
{
    const int q = par ^ 1, cm = pick4(c, mu), cn = pick4(c, nu);
    const int smu = up(g, s, cm, mu), snu = up(g, s, cn, nu), smd = dn(g, s, cm, mu), snd = dn(g, s, cn, nu);
    const int smd_nu = smd + (snu - s), smd_nd = smd + (snd - s), smu_nd = smu + (snd - s);
    Tri r{0.0, 0.0, 0.0, cd{0.0, 0.0}, cd{0.0, 0.0}, cd{0.0, 0.0}};
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    Raw6 a, b, k;
    ld_raw(U, g, s, mu, par, k);
    ld_raw(U, g, smu, nu, q, a);
    ld_raw(U, g, snu, mu, q, b);
    fence();
    // leaf I: U_mu(x) U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+
    M3 t = mul_r01(rows01(k), su3_of(a));
    ld_raw(U, g, s, nu, par, k);
    fence();
    t = mul_nd_r01(t, su3_of(b));
    ld_raw(U, g, smd_nu, mu, par, a);
    fence();
    t = mul_nd_r01(t, su3_of(k));
    ld_raw(U, g, smd, nu, q, b);
    fence();
    acc_leaf(r, t);
    retr = t.m[0].re + t.m[4].re + t.m[8].re;
    // leaf II: U_nu(x) U_mu(x-mu+nu)^+ U_nu(x-mu)^+ U_mu(x-mu)
    t = mul_nd_r01(rows01(k), su3_of(a));
    ld_raw(U, g, smd, mu, q, k);
    fence();
    t = mul_nd_r01(t, su3_of(b));
    ld_raw(U, g, smd_nd, nu, par, a);
    fence();
    t = mul_r01(t, su3_of(k));
    ld_raw(U, g, smd_nd, mu, par, b);
    fence();
    acc_leaf(r, t);
    // leaf III: U_mu(x-mu)^+ U_nu(x-mu-nu)^+ U_mu(x-mu-nu) U_nu(x-nu)
    t = mul_dd_r01(su3_of(k), su3_of(a));
    ld_raw(U, g, snd, nu, q, k);
    fence();
    t = mul_r01(t, su3_of(b));
    ld_raw(U, g, snd, mu, q, a);
    fence();
    t = mul_r01(t, su3_of(k));
    ld_raw(U, g, smu_nd, nu, par, b);
    fence();
    acc_leaf(r, t);
    // leaf IV: U_nu(x-nu)^+ U_mu(x-nu) U_nu(x+mu-nu) U_mu(x)^+
    t = mul_dn_r01(su3_of(k), su3_of(a));
    ld_raw(U, g, s, mu, par, k);
    fence();
    t = mul_r01(t, su3_of(b));
    t = mul_nd_r01(t, su3_of(k));
    acc_leaf(r, t);
    return r;
}
// Re tr(A B) of two anti-hermitian matrices in 9 reals
__device__ __forceinline__ double retr_ah(const Tri& a, const Tri& b)
{
    double d = a.d0 * b.d0;
    d = fma(a.d1, b.d1, d);
    d = fma(a.d2, b.d2, d);
    double o = a.r01.re * b.r01.re;
    o = fma(a.r01.im, b.r01.im, o);
    o = fma(a.r02.re, b.r02.re, o);
    o = fma(a.r02.im, b.r02.im, o);
    o = fma(a.r12.re, b.r12.re, o);
    o = fma(a.r12.im, b.r12.im, o);
    return -(d + 2.0 * o);
}
// directions of plane p in the order 01, 02, 03, 12, 13, 23.  Planes p and 5 - p are pair p
// (p < 3) of the topological charge tr R01 R23 - tr R02 R13 + tr R03 R12.
__device__ __forceinline__ int plane_mu(int p) { return p < 3 ? 0 : (p < 5 ? 1 : 2); }
__device__ __forceinline__ int plane_nu(int p) { return p < 3 ? p + 1 : (p < 5 ? p - 1 : 3); }
// The two planes of pair p at site s, each handed to take(plane, R, Re tr plaquette); returns
// the pair's term of the charge.  A loop, so that one plane at a time has the registers.
template <typename Take>
__device__ __forceinline__ double clover_pair(const double2* __restrict__ U, const Geom& g, int s, const int c[4], int par,
                                              int p, Take take)
{
    Tri first{};
    double q = 0.0;
#pragma unroll 1
    for (int j = 0; j < 2; ++j) {
        const int plane = j ? 5 - p : p;
        double pl;
        const Tri r = clover_ah(U, g, s, c, par, plane_mu(plane), plane_nu(plane), pl);
        take(plane, r, pl);
        if (j)
            q = retr_ah(first, r);
        else
            first = r;
    }
    return p == 1 ? -q : q;
}

// Derivative constants of the Cayley-Hamilton exponential (Morningstar-Peardon r_ij, b_ij
// with the sign-flip conjugation rules) from the closed form
__device__ __forceinline__ void exp_deriv_closed(const ExpC& e, ExpDeriv& out)
{
    const double u = e.u, u2 = e.u2, w2 = e.w2;
    const double xi0 = e.xi0, xi1 = xi1_of(e.w), cw = e.cosw;
    const cd em = e.exp_miu, e2 = e.exp_2iu;
    const cd ix = cd{0.0, xi0};
    const cd I = cd{0.0, 1.0};
    const cd f0 = e.denom * e.h0;
    const cd f1 = e.denom * e.h1, f2 = e.denom * e.h2;
    const cd r10 = 2.0 * (cd{u, u2 - w2} * e2)
                 + 2.0 * (em * ((4.0 * u) * cd{2.0, -u} * cw + ix * cd{9.0 * u2 + w2, -u * (3.0 * u2 + w2)}));
    const cd r11 = 2.0 * (cd{1.0, 2.0 * u} * e2) + em * (-2.0 * cd{1.0, -u} * cw + ix * cd{6.0 * u, w2 - 3.0 * u2});
    const cd r12 = 2.0 * (I * e2) + I * (em * (cd{cw, 0.0} - 3.0 * cd{1.0, -u} * xi0));
    const cd r20 = -2.0 * e2 + cd{0.0, 2.0 * u} * (em * (cd{cw, 0.0} + cd{1.0, 4.0 * u} * xi0 + cd{3.0 * u2 * xi1, 0.0}));
    const cd r21 = -(I * (em * (cd{cw, 0.0} + cd{1.0, 2.0 * u} * xi0 - cd{3.0 * u2 * xi1, 0.0})));
    const cd r22 = em * cd{xi0, -3.0 * u * xi1};
    cd b10, b11, b12, b20, b21, b22;
    if (e.c0max < 2.2250738585072014e-308) {
        b10 = b11 = b12 = b20 = b21 = b22 = cd{0.0, 0.0};
    } else {
        double bd = 9.0 * u2 - w2;
        bd *= 2.0 * bd;
        bd = 1.0 / bd;
        const double p = 3.0 * u2 - w2, q = 15.0 * u2 + w2;
        if (e.signflip) {
            b10 = bd * conj((2.0 * u) * r10 + p * r20 - (2.0 * q) * conj(f0));
            b11 = -bd * conj((2.0 * u) * r11 + p * r21 + (2.0 * q) * conj(f1));
            b12 = bd * conj((2.0 * u) * r12 + p * r22 - (2.0 * q) * conj(f2));
            b20 = -bd * conj(r10 - (3.0 * u) * r20 - (24.0 * u) * conj(f0));
            b21 = bd * conj(r11 - (3.0 * u) * r21 + (24.0 * u) * conj(f1));
            b22 = -bd * conj(r12 - (3.0 * u) * r22 - (24.0 * u) * conj(f2));
        } else {
            b10 = bd * ((2.0 * u) * r10 + p * r20 - (2.0 * q) * f0);
            b11 = bd * ((2.0 * u) * r11 + p * r21 - (2.0 * q) * f1);
            b12 = bd * ((2.0 * u) * r12 + p * r22 - (2.0 * q) * f2);
            b20 = bd * (r10 - (3.0 * u) * r20 - (24.0 * u) * f0);
            b21 = bd * (r11 - (3.0 * u) * r21 - (24.0 * u) * f1);
            b22 = bd * (r12 - (3.0 * u) * r22 - (24.0 * u) * f2);
        }
    }
    out = ExpDeriv{f0, f1, f2, b10, b11, b12, b20, b21, b22};
}
// f1, f2 and the b_ij of exp(iQ) from c0 = det Q, c1 = tr(Q^2)/2
__device__ __forceinline__ void exp_deriv(double c0, double c1, ExpDeriv& d)
{
    if (c1 <= EXP_SERIES_C1) {
        exp_series_deriv<EXP_TERMS>(c0, c1, d);
    } else {
        ExpC e;
        exp_constants_c(c0, c1, e);
        exp_deriv_closed(e, d);
    }
}

}  // namespace lt
