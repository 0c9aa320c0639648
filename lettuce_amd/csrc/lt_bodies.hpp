// lt_bodies.hpp -- per-thread bodies of the HMC and collective-variable kernels.
// Single-lattice kernels and the replica-batched kernels call the same bodies;
// link bodies take the logical block index b of their lattice (8 consecutive
// blocks = the (mu, parity) classes of one tile), site bodies take the site.
#pragma once

#include "lt_device.hpp"

// the MetaD stout tape kernel with the software-pipelined staple
#ifndef LT_MD_PIPE
#define LT_MD_PIPE 1
#endif

namespace lt {

// ---------------------------------------------------------------- HMC

// Momenta are anti-hermitian and traceless wherever the trajectory functions made them, and
// are kept in 8 reals then (ALG: ld_ah8, st_ah8, the first four of the nine slots): 64 bytes a
// link instead of 144.  The momenta a caller hands over are general matrices.

// P = 1/2 * A with A the anti-hermitian combination of the eight generators used
// by the reference's RandomMomentum; phi_1..phi_8 come from Philox stream
// RNG_MOMENTUM, draw blocks k = 0..3 (Box-Muller pairs).
template <bool ALG>
__device__ __forceinline__ void body_momentum(double2* __restrict__ P, const Geom& g, const LinkMap& m, int b,
                                              uint64_t seed, uint64_t counter)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    double phi[9];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        double u0, u1, g0, g1;
        draw2(seed, (uint32_t)s, RNG_MOMENTUM, (uint32_t)k, 0u, (uint32_t)mu, counter, u0, u1);
        gauss2(u0, u1, g0, g1);
        phi[1 + 2 * k] = g0;
        phi[2 + 2 * k] = g1;
    }
    const double s3 = sqrt(3.0);
    M3 A;
    A.m[0] = cd{0.0, phi[3] + phi[8] / s3};
    A.m[1] = cd{phi[2], phi[1]};
    A.m[2] = cd{phi[5], phi[4]};
    A.m[3] = cd{-phi[2], phi[1]};
    A.m[4] = cd{0.0, -phi[3] + phi[8] / s3};
    A.m[5] = cd{phi[7], phi[6]};
    A.m[6] = cd{-phi[5], phi[4]};
    A.m[7] = cd{-phi[7], phi[6]};
    A.m[8] = cd{0.0, -2.0 * phi[8] / s3};
    A = scale(0.5, A);
    if (ALG)
        st_ah8(P, g, s, mu, par, ah_tri(A));
    else
        st_link(P, g, s, mu, par, A);
}

// x += a y
__device__ __forceinline__ void axpy_tri(Tri& x, double a, const Tri& y)
{
    x.d0 += a * y.d0;
    x.d1 += a * y.d1;
    x.r01 += a * y.r01;
    x.r02 += a * y.r02;
    x.r12 += a * y.r12;
}

// P += a * Algebra(st U^+) + bf * F   (F optional: metadynamics force, whole matrices)
template <bool ALG>
__device__ __forceinline__ void body_force_update(const double2* __restrict__ U, double2* __restrict__ P,
                                                  const double2* __restrict__ F, const Geom& g, const LinkMap& m, int b,
                                                  double a, double bf)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    // 16^3 x 32, whole matrices: 60.8 us a launch, 63 with the plain staple
    Raw6 own;
    const M3 st = staple_pipelined(U, g, s, c, mu, par, own);
    M3 A = algebra(mul_nd(st, su3_of(own)));
    if (ALG) {
        Raw4 r;
        ld_ah8(P, g, s, mu, par, r);
        Tri p = her_of(r);
        axpy_tri(p, a, ah_tri(A));
        if (F) axpy_tri(p, bf, ah_tri(ld(F, g, s, mu, par)));
        st_ah8(P, g, s, mu, par, p);
        return;
    }
    M3 p = ld(P, g, s, mu, par);
    if (F) {
        M3 f = ld(F, g, s, mu, par);
#pragma unroll
        for (int k = 0; k < 9; ++k) p.m[k] += a * A.m[k] + bf * f.m[k];
    } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) p.m[k] += a * A.m[k];
    }
    st_link(P, g, s, mu, par, p);
}

// U <- exp(eps P) U, Gram-Schmidt (local per link, in place)
template <bool ALG>
__device__ __forceinline__ void body_field_update(double2* __restrict__ U, const double2* __restrict__ P, const Geom& g,
                                                  const LinkMap& m, int b, double eps)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    M3 E;
    if (ALG) {
        Raw4 r;
        ld_ah8(P, g, s, mu, par, r);
        const Tri p = her_of(r);
        E = exp_alg8(Alg8{p.d0, p.d1, p.r01, p.r02, p.r12}, eps);
    } else {
        E = exp_ah(ld(P, g, s, mu, par), eps);
    }
    M3 W = mul(E, ldu(U, g, s, mu, par));
    gram_schmidt(W);
    stu(U, g, s, mu, par, W);
}

// -Re tr(P P) of entry i of the 8 Vh entries (mu, parity, cb): lanes walk one array, and no
// coordinates are needed (one lane per (site, mu) in lexicographic order takes four times the
// L1 accesses; 16^3 x 32: 16.5 -> 15 us between events, the launch itself about 6)
template <bool ALG>
__device__ __forceinline__ double body_kinetic_link(const double2* __restrict__ P, const Geom& g, int i)
{
    const int a = i / g.Vh;
    const double2* q = P + slot_base(g, a, 9, i - a * g.Vh);
    if (ALG) {
        Raw4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r.v[e] = q[(size_t)e * slot_stride(g)];
        const Tri p = her_of(r);
        return -retr_ah(p, p);
    }
    M3 p;
#pragma unroll
    for (int e = 0; e < 9; ++e) p.m[e] = cd{q[(size_t)e * slot_stride(g)].x, q[(size_t)e * slot_stride(g)].y};
    return -retr_mul(p, p);
}

// entry i of the 8 Vh entries: P += a F with P in 8 reals and F whole matrices, or (a = 0, no
// F) P written out as whole matrices
template <bool WHOLE>
__device__ __forceinline__ void body_momentum_entry(double2* __restrict__ P, const double2* __restrict__ F, const Geom& g,
                                                    int i, double a)
{
    const int k = i / g.Vh;
    const size_t o = slot_base(g, k, 9, i - k * g.Vh), st = slot_stride(g);
    double2* q = P + o;
    if (WHOLE) {
        Raw4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r.v[e] = q[(size_t)e * st];
        const M3 p = add_ah(m3_zero(), her_of(r));
#pragma unroll
        for (int e = 0; e < 9; ++e) q[(size_t)e * st] = make_double2(p.m[e].re, p.m[e].im);
    } else {
        const double2* f = F + o;
        q[0] = make_double2(q[0].x + a * f[0].y, q[0].y + a * f[4 * st].y);
#pragma unroll
        for (int e = 1; e < 4; ++e) {
            const double2 v = f[(size_t)(e == 3 ? 5 : e) * st];
            q[(size_t)e * st] = make_double2(q[(size_t)e * st].x + a * v.x, q[(size_t)e * st].y + a * v.y);
        }
    }
}

// ------------------------------------------------- collective variable

// plane index of (a, b), a < b: 01,02,03,12,13,23
__device__ __forceinline__ int plane_of(int a, int b)
{
    return a == 0 ? b - 1 : (a == 1 ? b + 1 : 5);
}

// The clover planes are kept as R_munu = C_munu - C_munu^+ (mu < nu), which is all
// the charge and its derivative use.  R is anti-hermitian: 9 reals stored exactly,
//   R[((plane*2 + parity)*5 + k)*Vh + cb],
//   k: 0 r01, 1 r02, 2 r12, 3 (Im r00, Im r11), 4 (Im r22, 0);
// Re r_ii = 0 and r_ji = -conj(r_ij) hold exactly for C - C^+ in floating point.
__device__ __forceinline__ Tri ld_plane_tri(const double2* __restrict__ R, const Geom& g, int s, int plane, int par)
{
    const double2* p = R + slot_base(g, plane * 2 + par, R_SLOTS, cbi(g, s));
    const double2 a01 = p[0], a02 = p[slot_stride(g)], a12 = p[(size_t)2 * slot_stride(g)];
    const double2 d01 = p[(size_t)3 * slot_stride(g)], d2 = p[(size_t)4 * slot_stride(g)];
    return Tri{d01.x, d01.y, d2.x, cd{a01.x, a01.y}, cd{a02.x, a02.y}, cd{a12.x, a12.y}};
}
__device__ __forceinline__ void st_plane(double2* __restrict__ R, const Geom& g, int s, int plane, int par, const Tri& r)
{
    double2* p = R + slot_base(g, plane * 2 + par, R_SLOTS, cbi(g, s));
    p[0] = make_double2(r.r01.re, r.r01.im);
    p[slot_stride(g)] = make_double2(r.r02.re, r.r02.im);
    p[(size_t)2 * slot_stride(g)] = make_double2(r.r12.re, r.r12.im);
    p[(size_t)3 * slot_stride(g)] = make_double2(r.d0, r.d1);
    p[(size_t)4 * slot_stride(g)] = make_double2(r.d2, 0.0);
}

// stout level with tape: Q = -i rho Algebra(st U^+), U' = exp(iQ) U, Gram-Schmidt.
// KEEP: the link read is also stored in keep, which keeps level 0 of a stack without a copy
// of the field beforehand (a template: tested at run time the branch cost 224 spilled VGPRs).
template <bool KEEP>
__device__ __forceinline__ void body_stout_tape(const double2* __restrict__ Uin, double2* __restrict__ Uout,
                                                double2* __restrict__ T, const Geom& g, const LinkMap& m, int b,
                                                double rho, double2* __restrict__ keep)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
#if LT_MD_PIPE
    Raw6 own;
    const M3 st = staple_pipelined(Uin, g, s, c, mu, par, own);
    const M3 L = su3_of(own);
#else
    M3 st = staple(Uin, g, s, c, mu);
    M3 L = ldu(Uin, g, s, mu, par);
#endif
    M3 A = algebra(mul_nd(st, L));
    M3 Q;
#pragma unroll
    for (int k = 0; k < 9; ++k) Q.m[k] = cd{rho * A.m[k].im, -rho * A.m[k].re};
    st_her8(T, g, s, mu, par, Q);
    M3 W = mul(exp_her(Tri{Q.m[0].re, Q.m[4].re, -(Q.m[0].re + Q.m[4].re), Q.m[1], Q.m[2], Q.m[5]}), L);
    if (KEEP) stu_stream(keep, g, s, mu, par, L);
    gram_schmidt(W);
    stu(Uout, g, s, mu, par, W);
}

// Planes p and 5 - p of the site of index i (half_cb order), stored, and their term of the
// charge density Re tr(R01 R23 - R02 R13 + R03 R12)
__device__ __forceinline__ double body_clover_pair(const double2* __restrict__ U, double2* __restrict__ C, const Geom& g,
                                                   int i, int p)
{
    const int cb = half_cb(i), par = half_par(i);
    if (cb >= g.Vh) return 0.0;
    int c[4];
    const int s = site_of_cb(g, cb, par, c);
    return clover_pair(U, g, s, c, par, p, [&](int plane, const Tri& r, double) { st_plane(C, g, s, plane, par, r); });
}

// Re tr of the plaquette U_mu(x) U_nu(x+mu) U_mu(x+nu)^+ U_nu(x)^+ (plaquette.hpp:20-24)
// as Re tr(A B^+) with A = U_mu(x) U_nu(x+mu), B = U_nu(x) U_mu(x+nu), both in SU(3), of
// which only rows 0 and 1 are multiplied out (retr_su3_nd_r01).
__device__ __forceinline__ double plaq_plane(const double2* __restrict__ U, const Geom& g, int s, const int c[4],
                                            int par, int mu, int nu)
{
    const int smu = up(g, s, pick4(c, mu), mu), snu = up(g, s, pick4(c, nu), nu);
    const M3 A = mul_r01(ldu2(U, g, s, mu, par), ldu(U, g, smu, nu, par ^ 1));
    const M3 B = mul_r01(ldu2(U, g, s, nu, par), ldu(U, g, snu, mu, par ^ 1));
    return retr_su3_nd_r01(A, B);
}
// Re tr of the plaquettes of planes p and 5 - p at the site of index i (half_cb order)
__device__ __forceinline__ double body_plaq_pair(const double2* __restrict__ U, const Geom& g, int i, int p)
{
    const int cb = half_cb(i), par = half_par(i);
    if (cb >= g.Vh) return 0.0;
    int c[4];
    const int s = site_of_cb(g, cb, par, c);
    return plaq_plane(U, g, s, c, par, plane_mu(p), plane_nu(p)) + plaq_plane(U, g, s, c, par, plane_mu(5 - p), plane_nu(5 - p));
}
// The plaquettes of link (x, mu) in a launch over the field's link map: the planes
// (mu, mu+1 mod 4) and, for mu < 2, (mu, mu+2) -- every plane of every site once -- in the
// tile order of the link kernels, so that the neighbour links a tile reads are still in
// the L2 when the neighbouring tiles read them.
__device__ __forceinline__ double body_plaq_link(const double2* __restrict__ U, const Geom& g, const LinkMap& m, int b)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return 0.0;
    double v = plaq_plane(U, g, s, c, par, mu, (mu + 1) & 3);
    if (mu < 2) v += plaq_plane(U, g, s, c, par, mu, mu + 2);
    return v;
}
// sum of v over a link-map block of n lanes into *out: a butterfly in each wavefront, then the
// wavefront sums in wave order (sh: LT_LINK_BS / 64 doubles).  A map's block may end in a part of
// a wavefront (96 lanes for whole rows of 24 z): such a kernel is launched with whole ones
// (sum_block), whose further lanes have no site and bring zero.
__device__ __forceinline__ void link_block_sum(double v, int n, double* sh, double* out)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < ((n + 63) >> 6); ++w) v += sh[w];
        *out = v;
    }
}
// block sums of body_plaq_link, part[blockIdx.x]
__device__ __forceinline__ void plaq_link_partials(const double2* __restrict__ U, const Geom& g, const LinkMap& m,
                                                   double* part)
{
    __shared__ double sh[LT_LINK_BS / 64];
    link_block_sum(body_plaq_link(U, g, m, link_block(m, blockIdx.x, gridDim.x)), m.nthreads, sh, part + blockIdx.x);
}

// Running sums in LDS (entries e * n of a per-lane slot, e < 9): a sum waits there between the
// directions, so that one half term at a time has the registers; the empty asm statements with
// memory clobbers keep the compiler from carrying it in registers anyway.
template <int SG>
__device__ __forceinline__ void park_acc(double2* slot, int n, const M3& a)
{
    asm volatile("" ::: "memory");
#pragma unroll
    for (int e = 0; e < 9; ++e) {
        const double2 o = slot[e * n];
        slot[e * n] = SG > 0 ? make_double2(o.x + a.m[e].re, o.y + a.m[e].im)
                             : make_double2(o.x - a.m[e].re, o.y - a.m[e].im);
    }
    asm volatile("" ::: "memory");
}

// Clover-charge derivative for link (x, mu) (CloverDerivativeComponent,
// LettuceGauge/observables/clover.hpp:238-321): for each of the three nu != mu, with (rho,
// sigma) the remaining directions, R their clover plane and s = eps(mu, nu, rho, sigma), the
// reference's eight products per half regroup to
//   upper = S R(x) + R(x+mu) S + c (b^+ R(x+nu) + R(x+mu+nu) b^+) a^+,  S = c b^+ a^+
//   lower = T R(x) + R(x+mu) T + f^+ (e^+ R(x-nu) + R(x+mu-nu) e^+) d,  T = f^+ e^+ d
// with a = U_nu(x), b = U_mu(x+nu), c = U_nu(x+mu), d = U_nu(x-nu), e = U_mu(x-nu),
// f = U_nu(x+mu-nu), so that the terms with R(x) and R(x+mu) are taken once, of S - T, and
// the staples S, T are SU(3) matrices of which two rows are multiplied out.  The sum of
// s (upper - lower) over nu ends with
//   F(x, mu) = scale * (-2/(512 pi^2)) Algebra(U_mu(x) * sum).
// The running sum waits in LDS, as do S's two rows while the lower half is formed.  About
// 1500 FP64 instructions per nu instead of 1900.
// LDS: 15 x 16 bytes per lane of the block.
constexpr int CDERIV_SLOTS = 15;
__device__ __forceinline__ void lambda_link(const M3& sig, const Tri& Q, double2* __restrict__ Sig,
                                            double2* __restrict__ Lam, const Geom& g, int s, int mu, int par);
// LAMBDA: the force is the Sigma of the top stout level; instead of storing it the kernel
// goes on with that level's Lambda (lambda_link, next: its tape and the Lambda buffer), as the
// first launch of the stout-force recursion would.
template <bool LAMBDA>
__device__ __forceinline__ void body_clover_deriv_all(const double2* __restrict__ U, const double2* __restrict__ C,
                                                      double2* __restrict__ F, const Geom& g, const LinkMap& m, int b,
                                                      double scale_factor, double2* lds, const SigmaNext& next)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    const int n = m.nthreads, q = par ^ 1;
    double2* sum = lds + threadIdx.x;
    double2* wait = sum + 9 * n;
    park_store(sum, n, m3_zero());
    const int smu = up(g, s, pick4(c, mu), mu);
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        const int nu = k < mu ? k : k + 1;
        const int rho = (mu != 0 && nu != 0) ? 0 : ((mu != 1 && nu != 1) ? 1 : 2);
        const int sigma = (mu != 3 && nu != 3) ? 3 : ((mu != 2 && nu != 2) ? 2 : 1);
        const int inv = (mu > nu) + (mu > rho) + (mu > sigma) + (nu > rho) + (nu > sigma) + (rho > sigma);
        const double sign = (inv & 1) ? -1.0 : 1.0;
        const int plane = plane_of(rho, sigma);
        const int cnu = pick4(c, nu);
        {
            const int snu = up(g, s, cnu, nu);
            const M3 bd = dag(ldu(U, g, snu, mu, q));
            const M3 cc = ldu(U, g, smu, nu, q);
            const M3 a = ldu(U, g, s, nu, par);
            const M3 S = mul_nd_r01(mul_r01(cc, bd), a);
            asm volatile("" ::: "memory");
#pragma unroll
            for (int e = 0; e < 6; ++e) wait[e * n] = make_double2(S.m[e].re, S.m[e].im);
            asm volatile("" ::: "memory");
            M3 K = m3_zero();
            mul_tri_acc<true, 1>(K, bd, ld_plane_tri(C, g, snu, plane, q));
            tri_mul_acc<true, 1>(K, ld_plane_tri(C, g, up(g, smu, cnu, nu), plane, par), bd);
            park_acc<1>(sum, n, scale(sign, mul_nd(mul(cc, K), a)));
        }
        {
            const int snd = dn(g, s, cnu, nu), smu_nd = dn(g, smu, cnu, nu);
            const M3 ed = dag(ldu(U, g, snd, mu, q));
            const M3 f = ldu(U, g, smu_nd, nu, par);
            const M3 d = ldu(U, g, snd, nu, q);
            M3 D = mul_r01(mul_dn_r01(f, ed), d);
            third_row(D);
            M3 K = m3_zero();
            mul_tri_acc<true, 1>(K, ed, ld_plane_tri(C, g, snd, plane, q));
            tri_mul_acc<true, 1>(K, ld_plane_tri(C, g, smu_nd, plane, par), ed);
            M3 X = mul(mul_dn(f, K), d);
            asm volatile("" ::: "memory");
            M3 S;
#pragma unroll
            for (int e = 0; e < 6; ++e) S.m[e] = cd{wait[e * n].x, wait[e * n].y};
            third_row(S);
            D = sub(D, S);   // T - S
            mul_tri_acc<true, 1>(X, D, ld_plane_tri(C, g, s, plane, par));
            tri_mul_acc<true, 1>(X, ld_plane_tri(C, g, smu, plane, q), D);
            park_acc<-1>(sum, n, scale(sign, X));
        }
    }
    M3 a = park_load(sum, n);
    const double pref = -2.0 / (512.0 * 3.14159265358979323846 * 3.14159265358979323846);
    const M3 L = ldu(U, g, s, mu, par);
    a = scale(scale_factor * pref, algebra(mul(L, a)));
    if (LAMBDA)
        lambda_link(a, ld_her8_tri(next.T, g, s, mu, par), F, next.Lam, g, s, mu, par);
    else
        st_link(F, g, s, mu, par, a);
}

// Lambda = TracelessHermitian(tr(B1 G) Q + tr(B2 G) Q^2 + f1 G + f2 (Q G + G Q)), G = U Sigma',
// Sigma' = Uprev^+ Sigma, of one link.  Uprev = exp(iQ) U and Sigma is anti-hermitian and
// traceless, so G = exp(-iQ) Sigma needs neither field, and what the level below adds to its
// own terms is U (Sigma' exp(iQ)) = exp(-iQ) Sigma exp(iQ) = Y, again anti-hermitian and
// traceless: Y goes to Sig in 8 reals.  Storing Sigma' (9 complex entries), reading it, the
// tape and the next level's links again and evaluating the exponential once more took 736
// bytes a link and level instead of 416, and about 10 % more FP64 instructions.
__device__ __forceinline__ void lambda_link(const M3& sig, const Tri& Q, double2* __restrict__ Sig,
                                            double2* __restrict__ Lam, const Geom& g, int s, int mu, int par)
{
    const Tri Q2 = her_square(Q);
    ExpDeriv d;
    exp_deriv(her_det(Q), 0.5 * (Q2.d0 + Q2.d1 + Q2.d2), d);
    const M3 E = her_poly(d.f0, d.f1, d.f2, Q, Q2);
    M3 G = m3_zero();
    mul_tri_acc<true, 1>(G, dag(E), ah_tri(sig));
    st_ah8(Sig, g, s, mu, par, mul_ah(G, E));
    M3 QG = m3_zero();   // Q G + G Q, of trace 2 tr(Q G)
    mul_tri_acc<false, 1>(QG, G, Q);
    tri_mul_acc<false, 1>(QG, Q, G);
    // tr(B_i G) = b_i0 tr G + b_i1 tr(Q G) + b_i2 tr(Q^2 G)
    const cd tg = trace(G), tqg = 0.5 * trace(QG);
    cd tq2g = Q2.d0 * G.m[0] + Q2.d1 * G.m[4] + Q2.d2 * G.m[8];
    cmul_acc<1>(tq2g, Q2.r01, G.m[3]);
    cmul_acc<1>(tq2g, Q2.r02, G.m[6]);
    cmul_acc<1>(tq2g, Q2.r12, G.m[7]);
    cmul_acc<1>(tq2g, conj(Q2.r01), G.m[1]);
    cmul_acc<1>(tq2g, conj(Q2.r02), G.m[2]);
    cmul_acc<1>(tq2g, conj(Q2.r12), G.m[5]);
    const cd t1 = d.b10 * tg + d.b11 * tqg + d.b12 * tq2g;
    const cd t2 = d.b20 * tg + d.b21 * tqg + d.b22 * tq2g;
    // traceless hermitian part of t1 Q + t2 Q^2 + f1 G + f2 (Q G + G Q): Q and Q^2 are
    // hermitian, so only the real parts of t1 and t2 stay
    M3 Gam;
#pragma unroll
    for (int k = 0; k < 9; ++k) Gam.m[k] = d.f1 * G.m[k] + d.f2 * QG.m[k];
    Gam.m[0].re += t1.re * Q.d0 + t2.re * Q2.d0;
    Gam.m[4].re += t1.re * Q.d1 + t2.re * Q2.d1;
    Gam.m[8].re += t1.re * Q.d2 + t2.re * Q2.d2;
    Gam = tl_herm(Gam);
    Gam.m[1] += t1.re * Q.r01 + t2.re * Q2.r01;
    Gam.m[2] += t1.re * Q.r02 + t2.re * Q2.r02;
    Gam.m[5] += t1.re * Q.r12 + t2.re * Q2.r12;
    st_her8(Lam, g, s, mu, par, Gam);
}
// Sigma as a whole matrix in Sig
__device__ __forceinline__ void body_lambda(double2* __restrict__ Sig, const double2* __restrict__ T,
                                            double2* __restrict__ Lam, const Geom& g, const LinkMap& m, int b)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    lambda_link(ld(Sig, g, s, mu, par), ld_her8_tri(T, g, s, mu, par), Sig, Lam, g, s, mu, par);
}

// The six-term sum and the staple st are formed in one loop over nu != mu from the same
// neighbour links, each waiting in LDS between the halves (fs at lds + lane, st after it:
// entries e * nthreads, e < 9), then the sigma update.  With a = U_nu(x), b = U_mu(x+nu),
// c = U_nu(x+mu), d = U_nu(x-nu), e = U_mu(x-nu), f = U_nu(x+mu-nu), t = a b c^+ and
// d^+ e f the two staple terms and L the Lambda fields, the reference's products regroup to
//   upper: t^+ L_nu(x) - L_nu(x+mu) t^+ + c b^+ L_mu(x+nu) a^+
//   lower: f^+ (e^+ (L_mu(x-nu) - L_nu(x-nu)) + L_nu(x+mu-nu) e^+) d
// The products with a Lambda use that it is hermitian (mul_tri_acc).  About 1250 FP64
// instructions per nu instead of 1450.
// LDS: 18 x 16 bytes per lane of the block.
// The level's Sigma is Y + i rho Algebra(U (st^+ Lambda - sum)), Y from lambda_link.
// Bound by load latency and VALU issue together at the two waves per SIMD that 246 registers
// and 288 bytes of LDS a lane leave: a wave alone needs 10 us of VALU issue and twice that in
// all, the first direction's halves longest (their lines come from beyond the L2).  b and its
// Lambda are loaded a half ahead, the link's own after the last half.  Between events, levels
// with a Lambda and the last one: 16 x 8^4 90 -> 84.7 us, 16^4 106 -> 98 us with Y instead of
// Sigma' and the early loads; loading every operand two products ahead spills 68 registers.
// Blocks of one wave (FORCE_BLOCK) take that to 78 and 80 us.
// MODE SIGMA_STORE stores the result in Sig.  SIGMA_LAMBDA goes on with the Lambda of the
// level below for the same link, with that level's tape and Lambda buffer in next (not the
// Lambda buffer this launch reads: other lanes still read their neighbours' entries there).
// SIGMA_KICK (the last level of the recursion inside a metadynamics momentum update): the
// result is the bias force at level 0, and instead of storing it the kernel applies
// UpdateMomenta to the link (momenta in 8 reals), P += a Algebra(st U^+) + bf * force, with the staple it
// already holds -- body_force_update's formula, without the force field's store and
// load and the staple formed again (the momenta agree with the separate update to
// rounding, not bit for bit: the products are contracted into fused multiply-adds
// differently).
enum SigmaMode { SIGMA_STORE = 0, SIGMA_KICK = 1, SIGMA_LAMBDA = 2 };
template <int MODE>
__device__ __forceinline__ void body_sigma_all(const double2* __restrict__ U, double2* __restrict__ Sig,
                                               const double2* __restrict__ Lam,
                                               const Geom& g, const LinkMap& m, int b, double rho, double2* lds,
                                               const MomentumKick& kick, const SigmaNext& next)
{
    int mu, par, c[4], s;
    if (!map_link_b(g, m, b, mu, par, c, s)) return;
    const int n = m.nthreads;
    double2* fs_slot = lds + threadIdx.x;
    double2* st_slot = fs_slot + 9 * n;
    park_store(fs_slot, n, m3_zero());
    park_store(st_slot, n, m3_zero());
    const int q = par ^ 1;
    const int smu = up(g, s, pick4(c, mu), mu);
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    Raw6 rb;
    Raw4 rl;
    int nu = mu == 0 ? 1 : 0, cnu = pick4(c, nu), snu = up(g, s, cnu, nu);
    ld_raw(U, g, snu, mu, q, rb);
    ld_raw4(Lam, g, snu, mu, q, rl);
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        const int snd = dn(g, s, cnu, nu);
        const int smu_nd = dn(g, smu, cnu, nu);
        {
            const M3 a = ldu(U, g, s, nu, par);
            const M3 cc = ldu(U, g, smu, nu, q);
            const M3 b = su3_of(rb);
            M3 K = m3_zero();
            mul_tri_acc<false, 1>(K, dag(b), her_of(rl));
            M3 t = mul_nd_r01(mul_r01(a, b), cc);   // staple, upper term
            third_row(t);
            park_acc<1>(st_slot, n, t);
            M3 X = mul_nd(mul(cc, K), a);
            fence();
            ld_raw(U, g, snd, mu, q, rb);            // e and its Lambda for the lower half
            ld_raw4(Lam, g, snd, mu, q, rl);
            fence();
            t = dag(t);
            mul_tri_acc<false, 1>(X, t, ld_her8_tri(Lam, g, s, nu, par));
            tri_mul_acc<false, -1>(X, ld_her8_tri(Lam, g, smu, nu, q), t);
            park_acc<1>(fs_slot, n, X);
        }
        {
            const M3 f = ldu(U, g, smu_nd, nu, par);
            const M3 d = ldu(U, g, snd, nu, q);
            const M3 e = su3_of(rb);
            M3 t = mul_r01(e, f);
            third_row(t);
            t = mul_dn_r01(d, t);                   // staple, lower term
            third_row(t);
            park_acc<1>(st_slot, n, t);
            const M3 ed = dag(e);
            M3 K = m3_zero();
            mul_tri_acc<false, 1>(K, ed, her_of(rl) - ld_her8_tri(Lam, g, snd, nu, q));
            tri_mul_acc<false, 1>(K, ld_her8_tri(Lam, g, smu_nd, nu, par), ed);
            fence();
            // the next direction's b and its Lambda; after the last one the link's own
            if (k < 2) {
                nu = k + 1 < mu ? k + 1 : k + 2;
                cnu = pick4(c, nu);
                snu = up(g, s, cnu, nu);
            }
            const int sn = k < 2 ? snu : s, pn = k < 2 ? q : par;
            ld_raw(U, g, sn, mu, pn, rb);
            ld_raw4(Lam, g, sn, mu, pn, rl);
            fence();
            park_acc<1>(fs_slot, n, mul(mul_dn(f, K), d));
        }
    }
    Raw4 y;
    ld_ah8(Sig, g, s, mu, par, y);
    Raw4 tape, p;
    if (MODE == SIGMA_LAMBDA) ld_raw4(next.T, g, s, mu, par, tape);
    if (MODE == SIGMA_KICK) ld_ah8(kick.P, g, s, mu, par, p);
    fence();
    M3 cl = m3_zero();   // st^+ Lambda - the six-term sum
    mul_tri_acc<false, 1>(cl, dag(park_load(st_slot, n)), her_of(rl));
    cl = sub(cl, park_load(fs_slot, n));
    const M3 L = su3_of(rb);
#pragma unroll
    for (int e = 0; e < 9; ++e) cl.m[e] = cd{-rho * cl.m[e].im, rho * cl.m[e].re};
    const M3 sig = add_ah(algebra(mul(L, cl)), her_of(y));
    if (MODE == SIGMA_STORE) {
        st_link(Sig, g, s, mu, par, sig);
    } else if (MODE == SIGMA_LAMBDA) {
        lambda_link(sig, her_of(tape), Sig, next.Lam, g, s, mu, par);
    } else {
        const M3 A = algebra(mul_nd(park_load(st_slot, n), L));
        Tri q8 = her_of(p);
        axpy_tri(q8, kick.a, ah_tri(A));
        axpy_tri(q8, kick.bf, ah_tri(sig));
        st_ah8(kick.P, g, s, mu, par, q8);
    }
}

}  // namespace lt
