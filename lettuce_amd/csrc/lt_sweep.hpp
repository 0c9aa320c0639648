// lt_sweep.hpp -- per-link bodies of the local updates, shared by the
// two-colour kernels (lt_update.hip) and the four-colour kernels (lt_cb4.hip):
// SU(2)-subgroup extraction and embedding, overrelaxation, the Kennedy-Pendleton /
// Fabricius-Haan heatbath sampler with Philox draws, the Checkerboard4 site map and
// the link update, several wavefronts per 64 links, with the Wilson or the rectangular staple.
#pragma once

#include "lt_device.hpp"

namespace lt {

struct SU2 {
    cd e11, e12;
};

__device__ __forceinline__ SU2 su2_mul(SU2 a, SU2 b)
{
    return SU2{a.e11 * b.e11 - mul_c(a.e12, b.e12), a.e11 * b.e12 + mul_c(a.e12, b.e11)};
}
__device__ __forceinline__ double su2_det(SU2 a)
{
    return a.e11.re * a.e11.re + a.e11.im * a.e11.im + a.e12.re * a.e12.re + a.e12.im * a.e12.im;
}

// SU(2) part of (L * st^+) restricted to rows/cols (i,j)
__device__ __forceinline__ SU2 extract(const M3& L, const M3& st, int i, int j)
{
    cd wii = mul_c(L.m[3 * i], st.m[3 * i]) + mul_c(L.m[3 * i + 1], st.m[3 * i + 1]) + mul_c(L.m[3 * i + 2], st.m[3 * i + 2]);
    cd wij = mul_c(L.m[3 * i], st.m[3 * j]) + mul_c(L.m[3 * i + 1], st.m[3 * j + 1]) + mul_c(L.m[3 * i + 2], st.m[3 * j + 2]);
    cd wji = mul_c(L.m[3 * j], st.m[3 * i]) + mul_c(L.m[3 * j + 1], st.m[3 * i + 1]) + mul_c(L.m[3 * j + 2], st.m[3 * i + 2]);
    cd wjj = mul_c(L.m[3 * j], st.m[3 * j]) + mul_c(L.m[3 * j + 1], st.m[3 * j + 1]) + mul_c(L.m[3 * j + 2], st.m[3 * j + 2]);
    return SU2{0.5 * (wii + conj(wjj)), 0.5 * (wij - conj(wji))};
}

// rows i and j of L <- embed(X) * L
__device__ __forceinline__ void embed_mul(M3& L, SU2 X, int i, int j)
{
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        cd a = L.m[3 * i + n], b = L.m[3 * j + n];
        L.m[3 * i + n] = X.e11 * a + X.e12 * b;
        L.m[3 * j + n] = conj(X.e11) * b - conj(X.e12) * a;
    }
}

__device__ __forceinline__ SU2 overrelax(SU2 A)
{
    double an = 1.0 / sqrt(su2_det(A));
    SU2 V{an * A.e11, an * A.e12};
    SU2 VV = su2_mul(V, V);
    return SU2{conj(VV.e11), -VV.e12};
}

// The draws of one Kennedy-Pendleton / Fabricius-Haan attempt k of the SU(2) sampler in the
// reference's draw order: Philox blocks 2k (r1, r2) and 2k+1 (r3, r0) of the site.  They do
// not depend on the link: y = log r1 + cos^2(2 pi r2) log r3, lambda^2 = coef * y.
__device__ __forceinline__ void kp_draw(uint64_t seed, uint32_t site, uint32_t sub, uint32_t mu, uint64_t counter, int k,
                                        double& y, double& r0)
{
    double ua0, ua1, ub0, ub1;
    draw2(seed, site, RNG_HEATBATH, (uint32_t)(2 * k), sub, mu, counter, ua0, ua1);
    draw2(seed, site, RNG_HEATBATH, (uint32_t)(2 * k + 1), sub, mu, counter, ub0, ub1);
    const double x1 = log(1.0 - ua0);
    const double x2 = cos(2.0 * 3.14159265358979323846 * (1.0 - ua1));
    const double x3 = log(1.0 - ub0);
    y = x1 + x2 * x2 * x3;
    r0 = ub1;
}
__device__ __forceinline__ bool kp_accept(double y, double r0, double coef, double& lambda_sq)
{
    lambda_sq = coef * y;
    return !(r0 * r0 + lambda_sq >= 1.0);
}
// One attempt; coef = -0.25 prefactor / sqrt(det A).  Returns whether it is accepted.
__device__ __forceinline__ bool kp_attempt(uint64_t seed, uint32_t site, uint32_t sub, uint32_t mu, uint64_t counter,
                                           int k, double coef, double& lambda_sq)
{
    double y, r0;
    kp_draw(seed, site, sub, mu, counter, k, y, r0);
    return kp_accept(y, r0, coef, lambda_sq);
}

// The direction of the accepted draw (Philox block 0xFFFFF): cos(theta), cos(phi), sin(phi)
__device__ __forceinline__ void kp_direction(uint64_t seed, uint32_t site, uint32_t sub, uint32_t mu, uint64_t counter,
                                             double& cos_theta, double& cp, double& sp)
{
    double phi, ct;
    draw2(seed, site, RNG_HEATBATH, 0xFFFFFu, sub, mu, counter, phi, ct);
    cos_theta = 1.0 - 2.0 * ct;
    sincos(2.0 * 3.14159265358979323846 * phi, &sp, &cp);
}
// The accepted SU(2) draw X times V^+, V = A / sqrt(det A)
__device__ __forceinline__ SU2 kp_element(SU2 V, double lambda_sq, double cos_theta, double cp, double sp)
{
    double x0 = 1.0 - 2.0 * lambda_sq;
    double abs_x = sqrt(1.0 - x0 * x0);
    double vec_norm = abs_x * sqrt(1.0 - cos_theta * cos_theta);
    SU2 X{cd{x0, vec_norm * cp}, cd{vec_norm * sp, abs_x * cos_theta}};
    SU2 Vd{conj(V.e11), -V.e12};
    return su2_mul(X, Vd);
}
// Kennedy-Pendleton / Fabricius-Haan SU(2) sampler in the reference's draw order: the
// first accepted attempt k = 0, 1, ..., max_iter; after max_iter+1 rejected attempts
// the identity is taken.
constexpr int KP_MAX_ITER = 10;

// Site i in [0, V/4) of colour k of direction mu under Checkerboard4, where the colour
// is (t + x + y + z + x_mu) mod 4 (iterators.hpp:141-169; extents divisible by 4):
//   mu != z: every (t, x, y) row holds Nz/4 of them, every fourth z starting at
//            (k - t - x - y - x_mu) mod 4;
//   mu == z: the colour is (t + x + y + 2z) mod 4, so only rows with t + x + y = k mod 2
//            hold any, Nz/2 each, every second z.
// One thread per site of the class; consecutive threads walk z, then y, x, t.
__device__ __forceinline__ bool cb4_site(const Geom& g, int mu, int k, int i, int c[4], int& s)
{
    if (i >= (g.V >> 2)) return false;
    if (mu != 3) {
        int row = div_by(4 * i, g.dz);
        const int j = i - row * (g.L[3] >> 2);
        c[2] = mod_div(row, g.dy);
        c[1] = mod_div(row, g.dx);
        c[0] = row;
        c[3] = ((k - c[0] - c[1] - c[2] - pick4(c, mu)) & 3) + 4 * j;
    } else {
        const int row = div_by(2 * i, g.dz);
        const int j = i - row * (g.L[3] >> 1);
        int plane = div_by(2 * row, g.dy);
        const int yh = row - plane * (g.L[2] >> 1);
        c[1] = mod_div(plane, g.dx);
        c[0] = plane;
        c[2] = 2 * yh + ((k - c[0] - c[1]) & 1);
        c[3] = (((k - c[0] - c[1] - c[2]) & 3) >> 1) + 2 * j;
    }
    s = ((c[0] * g.L[1] + c[1]) * g.L[2] + c[2]) * g.L[3] + c[3];
    return true;
}

// The part of Rectangular<R>::Staple (rectangular_action.hpp:103-242) of link (x, mu) that
// lies on one side (UP: +nu, else -nu) of one direction nu: the plaquette term and its
// three 1x2 rectangles.  With a, b, c the three links of the plaquette term (a b c^+ above,
// a^+ b c below, x' = x - nu) each rectangle replaces one of them by its own three-link
// staple:
//   above: (c_p a b + c_r (Va b + a Vb)) c^+ + c_r a b Vc^+
//     Va = U_mu(x-mu)^+ U_nu(x-mu) U_mu(x-mu+nu),  Vb = U_nu(x+nu) U_mu(x+2nu) U_nu(x+mu+nu)^+,
//     Vc^+ = U_mu(x+mu+nu) U_nu(x+2mu)^+ U_mu(x+mu)^+
//   below: (c_p a^+ b + c_r (Va^+ b + a^+ Vb)) c + c_r a^+ b Vc
//     Va^+ = U_mu(x-mu)^+ U_nu(x'-mu)^+ U_mu(x'-mu),  Vb = U_nu(x'-nu)^+ U_mu(x'-nu) U_nu(x'+mu-nu),
//     Vc = U_mu(x'+mu) U_nu(x'+2mu) U_mu(x+mu)^+
// Eleven products instead of fourteen; every product but the last is a chain of links, an
// SU(3) matrix, of which rows 0 and 1 are carried.  Each link is loaded while the product
// before it is formed; the scheduling barriers keep the compiler from hoisting all twelve
// link loads (which spills).
template <bool UP, bool RECT>
__device__ __forceinline__ M3 staple_action_side(const double2* __restrict__ U, const Geom& g, int s, const int c[4],
                                                 int mu, int nu, int par, double c_plaq, double c_rect)
{
    const int q = par ^ 1;
    constexpr int sg = UP ? 1 : -1;
    auto at = [&](int a, int b) { return shift2(g, s, c, mu, a, nu, b); };
    auto step = [&](int site, int dir, int parity, Raw6& into) {
        ld_raw(U, g, site, dir, parity, into);
        __builtin_amdgcn_sched_barrier(0);
    };
    Raw6 l0, l1;
    M3 ab, t, r;
    // rows 0 and 1 of a^(+) b, and of a^(+) Vb's first product
    {
        Raw6 a;
        ld_raw(U, g, UP ? s : at(0, -1), nu, UP ? par : q, a);
        step(at(0, sg), mu, q, l0);
        step(at(0, UP ? 1 : -2), nu, UP ? q : par, l1);
        ab = UP ? mul_r01(rows01(a), su3_of(l0)) : mul_dn_r01(su3_of(a), su3_of(l0));
        if (!RECT) {
            ld_raw(U, g, at(1, UP ? 0 : -1), nu, UP ? q : par, l0);
            t = UP ? mul_nd_r01(ab, su3_of(l0)) : mul_r01(ab, su3_of(l0));
            third_row(t);
            return scale(c_plaq, t);
        }
        step(at(0, 2 * sg), mu, par, l0);
        t = UP ? mul_r01(rows01(a), su3_of(l1)) : mul_dd_r01(su3_of(a), su3_of(l1));
    }
    step(at(1, UP ? 1 : -2), nu, UP ? par : q, l1);
    t = mul_r01(t, su3_of(l0));
    step(at(-1, 0), mu, q, l0);
    t = UP ? mul_nd_r01(t, su3_of(l1)) : mul_r01(t, su3_of(l1));
    // Va^(+) b
    step(at(-1, UP ? 0 : -1), nu, UP ? q : par, l1);
    {
        const M3 d = su3_of(l0);
        step(at(-1, sg), mu, par, l0);
        r = UP ? mul_dn_r01(d, su3_of(l1)) : mul_dd_r01(d, su3_of(l1));
    }
    step(at(0, sg), mu, q, l1);
    r = mul_r01(r, su3_of(l0));
    step(at(1, UP ? 0 : -1), nu, UP ? q : par, l0);
    r = mul_r01(r, su3_of(l1));
    // (c_p a^(+) b + c_r (a^(+) Vb + Va^(+) b)) c^(+)
    M3 M = ab;
    third_row(M);
    third_row(t);
    acc_su3_r01(t, r);
#pragma unroll
    for (int e = 0; e < 9; ++e) M.m[e] = c_plaq * M.m[e] + c_rect * t.m[e];
    step(at(1, sg), mu, par, l1);
    M = UP ? mul_nd(M, su3_of(l0)) : mul(M, su3_of(l0));
    // a^(+) b Vc^(+)
    step(at(2, UP ? 0 : -1), nu, UP ? par : q, l0);
    r = mul_r01(ab, su3_of(l1));
    step(at(1, 0), mu, q, l1);
    r = UP ? mul_nd_r01(r, su3_of(l0)) : mul_r01(r, su3_of(l0));
    __builtin_amdgcn_sched_barrier(0);
    r = mul_nd_r01(r, su3_of(l1));
    third_row(r);
#pragma unroll
    for (int e = 0; e < 9; ++e) M.m[e] += c_rect * r.m[e];
    return M;
}

// Rectangular<R>::Staple (rectangular_action.hpp:232-242) of one link in one lane
template <bool RECT>
__device__ __forceinline__ M3 staple_action(const double2* __restrict__ U, const Geom& g, int s, const int c[4], int mu,
                                            int par, double c_plaq, double c_rect)
{
    M3 st = m3_zero();
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
        const int nu = k + (k >= mu);
        acc(st, staple_action_side<true, RECT>(U, g, s, c, mu, nu, par, c_plaq, c_rect));
        acc(st, staple_action_side<false, RECT>(U, g, s, c, mu, nu, par, c_plaq, c_rect));
    }
    return st;
}

// A colour launch with the staple split over wavefronts.  A block of WAVES wavefronts updates
// 64 links: wavefront w forms the part of the staple of the w-th direction nu != mu (WAVES = 3)
// or of side w & 1 of the (w >> 1)-th one (6); the parts are added through LDS and the first
// wavefront applies the SU(2) steps.  The heatbath's random numbers do not depend on the link:
// the wavefronts also draw the first two attempts and the direction of the three subgroups
// while the links of their parts are on the way; only the rare third attempts are drawn in the
// SU(2) steps.  One lane per link holds a whole SIMD's registers at two wavefronts and runs
// 5000 instructions in a row.
// The action enters through the staple only (heatbath.hpp:110-129, overrelaxation.hpp:91-116):
// SPLIT_WILSON, SPLIT_SCALED (c_plaq times the plaquette staple), SPLIT_RECT.
enum SplitKind { SPLIT_WILSON = 0, SPLIT_SCALED = 1, SPLIT_RECT = 2 };
// Wavefronts per SIMD.  Blocks of six go 2, 2, 1, 1 on the SIMDs of a compute unit, so two of
// them are resident only where four wavefronts fit a SIMD: overrelaxation with the plaquette
// staple, 123 registers (four colours at 28^4 55.6 us with 133 registers, 51.8 with 123).  The
// rectangle staple needs 188 without spills and has one block either way (24^4 84.5 -> 81.6
// us; its heatbath gains nothing and keeps three).  Blocks of three fill three per SIMD.
constexpr int split_eu(bool heatbath, int kind, int waves)
{
    return heatbath || waves == 3 ? 3 : kind == SPLIT_RECT ? 2 : 4;
}
template <bool HEATBATH, int WAVES>
struct SplitShared {
    double2 part[(WAVES == 6 ? 27 : 18) * SPLIT_LINKS];
    double draw[HEATBATH ? 21 * SPLIT_LINKS : 1];   // y, r0 of (subgroup, attempt); cos, cos, sin of the directions
};

// one side of the Wilson staple for one direction, rows 0 and 1 and the third from them
template <bool UP, typename Between>
__device__ __forceinline__ M3 staple_wilson_side(const double2* __restrict__ U, const Geom& g, int s, const int c[4],
                                                 int mu, int nu, int par, Between between)
{
    const int q = par ^ 1;
    const int x1 = UP ? s : shift2(g, s, c, mu, 0, nu, -1);
    Raw6 a, b, e;
    ld_raw(U, g, x1, nu, UP ? par : q, a);
    ld_raw(U, g, UP ? shift2(g, s, c, mu, 0, nu, 1) : x1, mu, q, b);
    ld_raw(U, g, shift2(g, s, c, mu, 1, nu, UP ? 0 : -1), nu, UP ? q : par, e);
    __builtin_amdgcn_sched_barrier(0);
    between();
    __builtin_amdgcn_sched_barrier(0);
    M3 t = UP ? mul_nd_r01(mul_r01(rows01(a), su3_of(b)), su3_of(e)) : mul_r01(mul_dn_r01(su3_of(a), su3_of(b)), su3_of(e));
    third_row(t);
    return t;
}

// on: whether this lane holds a link (s, mu) of the launch
template <bool HEATBATH, int KIND, int WAVES>
__device__ __forceinline__ void update_links_split(double2* __restrict__ U, const Geom& g, int mu, bool on, int s,
                                                   const int c[4], double prefactor, uint64_t seed, uint64_t counter,
                                                   double c_plaq, double c_rect, SplitShared<HEATBATH, WAVES>& sh)
{
    static_assert(WAVES == 6 || (WAVES == 3 && KIND != SPLIT_RECT), "no such split");
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    M3 st = m3_zero();
    int par = 0;
    auto draw_attempt = [&](int sub, int attempt) {
        double y, r0;
        kp_draw(seed, (uint32_t)s, (uint32_t)sub, (uint32_t)mu, counter, attempt, y, r0);
        const int slot = 2 * (sub + 3 * attempt);
        sh.draw[slot * SPLIT_LINKS + lane] = y;
        sh.draw[(slot + 1) * SPLIT_LINKS + lane] = r0;
    };
    auto draws = [&]() {
        if (HEATBATH) {
            draw_attempt(w % 3, w / 3);
            if (WAVES == 3) draw_attempt(w, 1);
            if (w < 3) {
                double ct, cp, sp;
                kp_direction(seed, (uint32_t)s, (uint32_t)w, (uint32_t)mu, counter, ct, cp, sp);
                sh.draw[(12 + 3 * w) * SPLIT_LINKS + lane] = ct;
                sh.draw[(13 + 3 * w) * SPLIT_LINKS + lane] = cp;
                sh.draw[(14 + 3 * w) * SPLIT_LINKS + lane] = sp;
            }
        }
    };
    if (on) {
        par = parity_of(c);
        const int d = WAVES == 6 ? w >> 1 : w, nu = d + (d >= mu);
        if (KIND == SPLIT_RECT) {
            draws();
            st = (w & 1) ? staple_action_side<false, true>(U, g, s, c, mu, nu, par, c_plaq, c_rect)
                         : staple_action_side<true, true>(U, g, s, c, mu, nu, par, c_plaq, c_rect);
        } else if (WAVES == 6) {
            st = (w & 1) ? staple_wilson_side<false>(U, g, s, c, mu, nu, par, draws)
                         : staple_wilson_side<true>(U, g, s, c, mu, nu, par, draws);
        } else {
            st = staple_wilson_side<true>(U, g, s, c, mu, nu, par, draws);
            acc(st, staple_wilson_side<false>(U, g, s, c, mu, nu, par, [] {}));
        }
        if (KIND == SPLIT_SCALED) st = scale(c_plaq, st);
    }
    auto put = [&](int slot) {
#pragma unroll
        for (int e = 0; e < 9; ++e) sh.part[(slot * 9 + e) * SPLIT_LINKS + lane] = make_double2(st.m[e].re, st.m[e].im);
    };
    auto add_from = [&](int slot) {
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            const double2 v = sh.part[(slot * 9 + e) * SPLIT_LINKS + lane];
            st.m[e] += cd{v.x, v.y};
        }
    };
    if (WAVES == 6) {
        if (w >= 3) put(w - 3);
        __syncthreads();
        if (w < 3) add_from(w);
        if (w == 1 || w == 2) put(w);
    } else if (w) {
        put(w - 1);
    }
    __syncthreads();
    if (w || !on) return;
    M3 L = ldu(U, g, s, mu, par);
    add_from(WAVES == 6 ? 1 : 0);
    add_from(WAVES == 6 ? 2 : 1);
#pragma unroll
    for (int sub = 0; sub < 3; ++sub) {
        const int i = sub == 2 ? 1 : 0;
        const int j = sub == 0 ? 1 : 2;
        // one subgroup at a time has the registers
        __builtin_amdgcn_sched_barrier(0);
        const SU2 A = extract(L, st, i, j);
        SU2 X;
        if (HEATBATH) {
            const double an = 1.0 / sqrt(su2_det(A));
            const SU2 V{an * A.e11, an * A.e12};
            const double coef = -0.25 * prefactor * an;
            const double* d = sh.draw + lane;
            double lambda_sq;
            bool found = kp_accept(d[2 * sub * SPLIT_LINKS], d[(2 * sub + 1) * SPLIT_LINKS], coef, lambda_sq);
            if (!found) found = kp_accept(d[(6 + 2 * sub) * SPLIT_LINKS], d[(7 + 2 * sub) * SPLIT_LINKS], coef, lambda_sq);
            for (int k = 2; !found && k <= KP_MAX_ITER; ++k)
                found = kp_attempt(seed, (uint32_t)s, (uint32_t)sub, (uint32_t)mu, counter, k, coef, lambda_sq);
            X = found ? kp_element(V, lambda_sq, d[(12 + 3 * sub) * SPLIT_LINKS], d[(13 + 3 * sub) * SPLIT_LINKS],
                                   d[(14 + 3 * sub) * SPLIT_LINKS])
                      : SU2{cd{1.0, 0.0}, cd{0.0, 0.0}};
        } else {
            X = overrelax(A);
        }
        embed_mul(L, X, i, j);
    }
    gram_schmidt(L);
    stu(U, g, s, mu, par, L);
}

// Index (in the class's order, t slowest) of the link of this lane in block b of a split
// launch; -1 for none.
__device__ __forceinline__ int split_index(const SplitMap& m, int b)
{
    int q = b;
    const int ch = div_by(b, m.dper);
    q -= ch * m.dper.d;
    const int t = mod_div(q, m.dtc);
    const int r = q * SPLIT_LINKS + (threadIdx.x & (SPLIT_LINKS - 1));
    return r < m.nt ? (ch * m.dtc.d + t) * m.nt + r : -1;
}

}  // namespace lt
