// lt_obs.hip -- fused observables pass: for every site the six clover terms C_munu
// (four leaves each) are built once and give the plaquette sum (leaf I is the
// plaquette), the clover topological-charge density and the clover energy
// density.  Reductions are deterministic: a fixed-shape block tree per timeslice
// chunk, then an ordered sum over chunks.
#include "lt_internal.hpp"
#include "lt_bodies.hpp"

#include <mutex>

namespace lt {

namespace {

constexpr int BS = 256;

// Re tr(f f) with f = traceless(-i/8 R), R anti-hermitian
__device__ __forceinline__ double energy_term(const Tri& r)
{
    const double t = (1.0 / 3.0) * (r.d0 + r.d1 + r.d2);
    const double a = r.d0 - t, b = r.d1 - t, c = r.d2 - t;
    const double o = r.r01.re * r.r01.re + r.r01.im * r.r01.im + r.r02.re * r.r02.re + r.r02.im * r.r02.im +
                     r.r12.re * r.r12.re + r.r12.im * r.r12.im;
    return (1.0 / 64.0) * (a * a + b * b + c * c + 2.0 * o);
}

__device__ __forceinline__ void block_sum3(double v0, double v1, double v2, double* out)
{
    double a[3] = {v0, v1, v2};
    block_reduce<BS>(a, OpAdd{});
    if (threadIdx.x == 0) {
        out[0] = a[0];
        out[1] = a[1];
        out[2] = a[2];
    }
}

// grid: 3 plane pairs x chunks per timeslice x Nt blocks, pair fastest, spread over the XCDs
// so each covers a contiguous range of timeslices with all three pairs of a chunk in
// neighbouring blocks (one L2-resident neighbourhood).  A lane takes planes p and 5 - p of one
// site (half_cb order within the timeslice), so the charge needs no exchange.  Sums of the
// plaquette, raw charge and energy of a block go to part[3 ((t nchunk + chunk) 3 + pair)].
// Bound by VALU issue (12 products and 13 links a plane) and load latency at the two waves per
// SIMD that 216 registers leave: 32^4 472 us.  Three waves spill 60 registers, whose reloads
// also wait for the links on the way (588 us); one lane per site with all six planes and the
// sums parked in LDS took 655 us, six waves for 64 sites 720 us.
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(2)))
obs_kernel(const double2* __restrict__ U, Geom g, int Vs, int nchunk, double* part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int pair = b % 3, tc = b / 3, t = tc / nchunk, chunk = tc - t * nchunk;
    const int i = chunk * BS + threadIdx.x, cb = half_cb(i), par = half_par(i);
    double p = 0.0, q = 0.0, e = 0.0;
    if (cb < (Vs >> 1)) {
        int c[4];
        const int s = site_of_cb(g, t * (Vs >> 1) + cb, par, c);
        q = clover_pair(U, g, s, c, par, pair, [&](int, const Tri& r, double pl) {
            p += pl;
            e += energy_term(r);
        });
    }
    block_sum3(p, q, e, part + 3 * (size_t)b);
}

// TopChargeClover's summand per site (topological_charge.hpp:184-199): one lane per site
// (half_cb order) evaluates all three plane pairs and writes, in lexicographic order,
// -1/(256 pi^2) (tr F01F23 - tr F02F13 + tr F03F12), F = C - C^+.
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(2)))
qdensity_kernel(const double2* __restrict__ U, Geom g, double* __restrict__ q_x)
{
    const int i = blockIdx.x * BS + threadIdx.x, cb = half_cb(i), par = half_par(i);
    if (cb >= g.Vh) return;
    int c[4];
    const int s = site_of_cb(g, cb, par, c);
    double q = 0.0;
#pragma unroll 1
    for (int p = 0; p < 3; ++p) q += clover_pair(U, g, s, c, par, p, [](int, const Tri&, double) {});
    q_x[s] = (-1.0 / (256.0 * M_PI * M_PI)) * q;
}

// one block per timeslice: lane i sums the entries i, i + BS, ... of its timeslice's 3 nchunk,
// then the block tree of block_sum3
__global__ void __launch_bounds__(BS) obs_finish_kernel(const double* part, int nchunk, int nt, double* out)
{
    const int t = blockIdx.x;
    double a = 0.0, b = 0.0, c = 0.0;
    for (int k = threadIdx.x; k < 3 * nchunk; k += BS) {
        const double* p = part + 3 * (3 * (size_t)t * nchunk + k);
        a += p[0];
        b += p[1];
        c += p[2];
    }
    block_sum3(a, b, c, out + 3 * (size_t)t);
}

// ---- the rest of Observables() (SU3_main.cpp:125-136) --------------------------

// neighbour of lexicographic site s with coordinates c, n steps along mu (|n| < L)
__device__ __forceinline__ int shift(const Geom& g, int s, const int c[4], int mu, int n)
{
    const int cm = pick4(c, mu);
    return s + (wrap_add(cm, n, pick4(g.L, mu)) - cm) * pick4(g.st, mu);
}

// Re tr of the plaquette (plaquette.hpp:20-24) and of the 1x2 and 2x1 loops
// (wilson_loop.hpp:155-175) of plane (mu, nu) at site s, each as Re tr(A B^+) of its two halves
// (chains of links, of which rows 0 and 1 are multiplied out).  Ten links (U_mu(x) twice), each
// loaded a product or two ahead.
__device__ __forceinline__ void plane_loops(const double2* __restrict__ U, const Geom& g, int s, const int c[4], int par,
                                            int mu, int nu, double& plaq, double& rect)
{
    const int q = par ^ 1;
    auto at = [&](int a, int b) { return shift2(g, s, c, mu, a, nu, b); };
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };
    Raw6 a, b, k;
    ld_raw(U, g, s, mu, par, a);
    ld_raw(U, g, at(1, 0), nu, q, b);
    ld_raw(U, g, s, nu, par, k);
    fence();
    // A = U_mu(x) U_nu(x+mu), B = U_nu(x) U_mu(x+nu): the plaquette is A B^+
    M3 A = mul_r01(rows01(a), su3_of(b));
    ld_raw(U, g, at(0, 1), mu, q, b);
    ld_raw(U, g, at(0, 1), nu, q, a);
    fence();
    M3 B = mul_r01(rows01(k), su3_of(b));
    ld_raw(U, g, at(0, 2), mu, par, b);
    fence();
    plaq = retr_su3_nd_r01(A, B);
    // 1x2: A U_nu(x+mu+nu) against U_nu(x) U_nu(x+nu) U_mu(x+2nu)
    M3 C = mul_r01(rows01(k), su3_of(a));
    ld_raw(U, g, at(1, 1), nu, par, k);
    fence();
    C = mul_r01(C, su3_of(b));
    ld_raw(U, g, at(1, 1), mu, par, a);
    fence();
    A = mul_r01(A, su3_of(k));
    ld_raw(U, g, s, mu, par, b);
    ld_raw(U, g, at(1, 0), mu, q, k);
    fence();
    rect = retr_su3_nd_r01(A, C);
    // 2x1: U_mu(x) U_mu(x+mu) U_nu(x+2mu) against B U_mu(x+mu+nu)
    B = mul_r01(B, su3_of(a));
    ld_raw(U, g, at(2, 0), nu, par, a);
    fence();
    C = mul_r01(rows01(b), su3_of(k));
    C = mul_r01(C, su3_of(a));
    rect += retr_su3_nd_r01(C, B);
}

__device__ __forceinline__ void block_sum2(double v0, double v1, double* out)
{
    double a[2] = {v0, v1};
    block_reduce<BS>(a, OpAdd{});
    if (threadIdx.x == 0) {
        out[0] = a[0];
        out[1] = a[1];
    }
}

// block k: the sum of part[K i + k], i < n (K = gridDim.x values per entry)
__global__ void __launch_bounds__(BS) sum_parts_kernel(const double* __restrict__ part, int n, double* out)
{
    block_sum_to<BS>(partials_sum<BS>(part + blockIdx.x, n, gridDim.x), out + blockIdx.x);
}

// grid: 3 plane pairs x ceil(V / BS) blocks, pair fastest, XCD-remapped; a lane takes planes p
// and 5 - p of one site (half_cb order).  Per block: sum Re tr P, sum Re tr (R12 + R21).
// Bound like obs_kernel: 32^4 395 us with 225 registers at two waves per SIMD (587 us with one
// lane per site and the plaquette charge beside it; 657 us at three waves, with spills).
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(2)))
rect_kernel(const double2* __restrict__ U, Geom g, double* part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int pair = b % 3, i = (b / 3) * BS + threadIdx.x, cb = half_cb(i), par = half_par(i);
    double p = 0.0, r = 0.0;
    if (cb < g.Vh) {
        int c[4];
        const int s = site_of_cb(g, cb, par, c);
#pragma unroll 1
        for (int j = 0; j < 2; ++j) {
            const int plane = j ? 5 - pair : pair;
            double pl, re;
            plane_loops(U, g, s, c, par, plane_mu(plane), plane_nu(plane), pl, re);
            p += pl;
            r += re;
        }
    }
    block_sum2(p, r, part + 2 * (size_t)b);
}

// TopChargePlaquette's summand (topological_charge.hpp:366-416): with F = -i (P - P^+) of the
// single plaquettes, Re tr (F01 F23 + F02 F31 + F03 F12) = -(tr D01 D23 - tr D02 D13 + tr D03 D12),
// D = P - P^+; grid and lanes as rect_kernel.  32^4 158 us, where the pass over the rectangles
// that it was part of took 587.
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(3)))
plaq_charge_kernel(const double2* __restrict__ U, Geom g, double* part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    const int pair = b % 3, i = (b / 3) * BS + threadIdx.x, cb = half_cb(i), par = half_par(i);
    double q = 0.0;
    if (cb < g.Vh) {
        int c[4];
        const int s = site_of_cb(g, cb, par, c);
        Tri first{};
#pragma unroll 1
        for (int j = 0; j < 2; ++j) {
            const int plane = j ? 5 - pair : pair, mu = plane_mu(plane), nu = plane_nu(plane);
            const int smu = up(g, s, pick4(c, mu), mu), snu = up(g, s, pick4(c, nu), nu);
            M3 t = mul_r01(ldu2(U, g, s, mu, par), ldu(U, g, smu, nu, par ^ 1));
            t = mul_nd_r01(t, ldu(U, g, snu, mu, par ^ 1));
            t = mul_nd_r01(t, ldu(U, g, s, nu, par));
            Tri r{};
            acc_leaf(r, t);
            if (j)
                q = -retr_ah(first, r);
            else
                first = r;
        }
        if (pair == 1) q = -q;
    }
    block_sum_to<BS>(q, part + b);
}

// WilsonLoop chain update (wilson_loop.hpp:71-88): chain(x, mu) <- [1 or chain(x, mu)]
// * U_mu(x + n0 mu) ... U_mu(x + (n1 - 1) mu), over the field's link map (lanes along one
// parity array; one lane per (site, mu) in memory order took four times the L1 accesses); the
// chains are streamed out.  Memory bound: 32^4, one link a call 365 -> 283 us (1.5 GB, 5.3 TB/s).
__global__ void LT_LINK_KERNEL wchain_kernel(const double2* __restrict__ U, double2* __restrict__ chain, Geom g, LinkMap m,
                                             int n0, int n1, int reset)
{
    int mu, par, c[4], s;
    if (!map_link_all(g, m, mu, par, c, s)) return;
    const int cm = pick4(c, mu), L = pick4(g.L, mu), st = pick4(g.st, mu);
    int v = (cm + n0 % L) % L;
    auto link = [&]() {
        const M3 u = ldu(U, g, s + (v - cm) * st, mu, (par + v + cm) & 1);
        v = v + 1 == L ? 0 : v + 1;
        return u;
    };
    int n = n0;
    M3 a;
    if (reset) {
        a = link();
        ++n;
    } else {
        a = ld(chain, g, s, mu, par);
    }
    for (; n < n1; ++n) a = mul(a, link());
    double2* p = chain + slot_base(g, mu * 2 + par, 9, cbi(g, s));
#pragma unroll
    for (int e = 0; e < 9; ++e) st_stream(p + (size_t)e * slot_stride(g), make_double2(a.m[e].re, a.m[e].im));
}

// the square loops of side L from the chains (wilson_loop.hpp:89-125):
// Re tr (chain_mu(x) chain_nu(x + L mu) (chain_nu(x) chain_mu(x + L nu))^+), the planes of a
// site spread over its links as for PlaquetteSum (body_plaq_link).  The chains are products of
// links, so in SU(3): rows 0 and 1 of each are read, rows 0 and 1 of both products multiplied
// out and the trace taken with retr_su3_nd_r01.  32^4 327 -> 180 us.
__global__ void LT_LINK_KERNEL wloop_kernel(const double2* __restrict__ chain, Geom g, LinkMap m, int L, double* part)
{
    __shared__ double sh[LT_LINK_BS / 64];
    int mu, par, c[4], s;
    double w = 0.0;
    if (map_link_all(g, m, mu, par, c, s)) {
        const int odd = L & 1;
        const int smu = shift(g, s, c, mu, L % pick4(g.L, mu));
#pragma unroll 1
        for (int k = 1; k < (mu < 2 ? 3 : 2); ++k) {
            const int nu = (mu + k) & 3, snu = shift(g, s, c, nu, L % pick4(g.L, nu));
            const M3 A = mul_r01(ldu2(chain, g, s, mu, par), ldu(chain, g, smu, nu, par ^ odd));
            const M3 B = mul_r01(ldu2(chain, g, s, nu, par), ldu(chain, g, snu, mu, par ^ odd));
            w += retr_su3_nd_r01(A, B);
        }
    }
    link_block_sum(w, m.nthreads, sh, part + blockIdx.x);
}

// PolyakovLoop (polyakov_loop.hpp:31-49): one lane per spatial site (half_cb order), tr prod_t U_t
__global__ void __launch_bounds__(BS) polyakov_kernel(const double2* __restrict__ U, Geom g, double* part)
{
    const int vs2 = (g.L[1] * g.L[2] * g.L[3]) >> 1;
    const int i = blockIdx.x * BS + threadIdx.x, cb = half_cb(i), par = half_par(i);
    double re = 0.0, im = 0.0;
    if (cb < vs2) {
        int c[4];
        int s = site_of_cb(g, cb, par, c);   // timeslice 0
        M3 a = m3_id();
        for (int t = 0; t < g.L[0]; ++t, s += g.st[0]) a = mul(a, ldu(U, g, s, 0, par ^ (t & 1)));
        re = a.m[0].re + a.m[4].re + a.m[8].re;
        im = a.m[0].im + a.m[4].im + a.m[8].im;
    }
    block_sum2(re, im, part + 2 * (size_t)blockIdx.x);
}

}  // namespace

namespace {

// the K sums of n entries of K partials each (they follow the partials in scratch)
void sum_parts(lt_ctx ctx, double* part, unsigned n, int K, double* out)
{
    double* fin = part + (size_t)K * n;
    launch(ctx, "sum_parts", sum_parts_kernel, dim3(K), dim3(BS), 0, (const double*)part, (int)n, fin);
    double* h = ctx->host_for(K);
    LT_HIP_CHECK(hipMemcpyAsync(h, fin, K * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    for (int k = 0; k < K; ++k) out[k] = h[k];
}

}  // namespace

// sums over sites of Re tr P and Re tr (R12 + R21)
void k_rect_sums(lt_field u, double out[2])
{
    lt_ctx ctx = u->ctx;
    const unsigned nb = 3 * nblocks(u->g.V, BS);
    double* part = ctx->scratch_for(2 * (size_t)nb + 2);
    launch(ctx, "rect", rect_kernel, dim3(nb), dim3(BS), 0, (const double2*)u->d, u->g, part);
    sum_parts(ctx, part, nb, 2, out);
}

// sum over sites of the raw plaquette charge density
double k_plaq_charge(lt_field u)
{
    lt_ctx ctx = u->ctx;
    const unsigned nb = 3 * nblocks(u->g.V, BS);
    double* part = ctx->scratch_for((size_t)nb + 1);
    launch(ctx, "plaq_charge", plaq_charge_kernel, dim3(nb), dim3(BS), 0, (const double2*)u->d, u->g, part);
    double q;
    sum_parts(ctx, part, nb, 1, &q);
    return q;
}

double k_wilson_loop(lt_field u, lt_field chain, int n0, int n1, int reset)
{
    lt_ctx ctx = u->ctx;
    const Geom& g = u->g;
    const LinkMap& m = u->map;
    const unsigned nb = 8 * map_blocks(m);
    launch(ctx, "wilson_chain", wchain_kernel, dim3(nb), dim3(m.nthreads), 0, (const double2*)u->d, chain->d, g, m, n0, n1,
           reset);
    double* part = ctx->scratch_for((size_t)nb + 1);
    launch(ctx, "wilson_loop", wloop_kernel, dim3(nb), sum_block(m), 0, (const double2*)chain->d, g, m, n1, part);
    double w;
    sum_parts(ctx, part, nb, 1, &w);
    return w;
}

void k_polyakov_loop(lt_field u, double* re, double* im)
{
    lt_ctx ctx = u->ctx;
    const Geom& g = u->g;
    const int vs = g.L[1] * g.L[2] * g.L[3];
    const unsigned nb = nblocks(vs, BS);
    double* part = ctx->scratch_for(2 * (size_t)nb + 2);
    launch(ctx, "polyakov_loop", polyakov_kernel, dim3(nb), dim3(BS), 0, (const double2*)u->d, g, part);
    double out[2];
    sum_parts(ctx, part, nb, 2, out);
    *re = out[0] / vs;
    *im = out[1] / vs;
}

void k_observables(lt_field u, double* host_out)
{
    lt_ctx ctx = u->ctx;
    const Geom& g = u->g;
    const int nt = g.L[0];
    const int Vs = g.V / nt;
    const unsigned nchunk = nblocks(Vs, BS);
    double* part = ctx->scratch_for(9 * (size_t)nchunk * nt + 3 * (size_t)nt);
    double* fin = part + 9 * (size_t)nchunk * nt;
    launch(ctx, "observables", obs_kernel, dim3(3 * nchunk * nt), dim3(BS), 0, (const double2*)u->d, g, Vs, (int)nchunk,
           part);
    launch(ctx, "observables_finish", obs_finish_kernel, dim3(nt), dim3(BS), 0, (const double*)part, (int)nchunk, nt,
           fin);
    LT_HIP_CHECK(hipMemcpyAsync(host_out, fin, 3 * (size_t)nt * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

// ---- observables without allocation ---------------------------------------------
// lt_observables_noalloc keeps its partial sums in this fixed device array instead of
// the context's scratch.  Host code uses only the per-device address that
// hipGetSymbolAddress returns (the array's name is a host-side stand-in).
namespace {

constexpr size_t NOALLOC_DOUBLES = (size_t)1 << 20;   // 8 MiB per GPU
constexpr int NOALLOC_MAX_DEVICES = 64;
__device__ __align__(256) double scratch[NOALLOC_DOUBLES];

std::mutex noalloc_mutex;
double* noalloc_ptr[NOALLOC_MAX_DEVICES] = {};

// The per-timeslice sums -> [plaq_sum, Q, E_plaq, E_clov, q_t[Nt], e_t[Nt]] in one
// thread, operation for operation as lt_observables does it on the host (no
// contraction), so both entry points return the same bits.
__global__ void obs_final_kernel(const double* __restrict__ h, int nt, double V, double* __restrict__ out)
{
#pragma clang fp contract(off)
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const double qnorm = -1.0 / (256.0 * M_PI * M_PI);
    double p = 0.0, q = 0.0, e = 0.0;
    for (int t = 0; t < nt; ++t) {
        const double qt = qnorm * h[3 * t + 1];
        const double et = h[3 * t + 2] / V;
        out[4 + t] = qt;
        out[4 + nt + t] = et;
        p += h[3 * t];
        q += qt;
        e += et;
    }
    out[0] = p;
    out[1] = q;
    out[2] = 2.0 * (18.0 - p / V);
    out[3] = e;
}

}  // namespace

void noalloc_setup(int device)
{
    if (device < 0 || device >= NOALLOC_MAX_DEVICES)
        throw LtError{LT_EINVAL, "device index beyond the fixed observables scratch table"};
    std::lock_guard<std::mutex> lock(noalloc_mutex);
    if (noalloc_ptr[device]) return;
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
        throw LtError{LT_EHIP, std::string("hipGetSymbolAddress(observables scratch): ") + hipGetErrorString(e)};
    noalloc_ptr[device] = (double*)p;
}

size_t noalloc_observables_doubles(const Geom& g)
{
    const int nt = g.L[0];
    const size_t nchunk = nblocks(g.V / nt, BS);
    return 9 * nchunk * nt + 3 * (size_t)nt + 4 + 2 * (size_t)nt;
}

void k_observables_noalloc(lt_field u, double* host_out)
{
    lt_ctx ctx = u->ctx;
    const Geom& g = u->g;
    const size_t need = noalloc_observables_doubles(g);
    if (need > NOALLOC_DOUBLES)
        throw LtError{LT_EINVAL, "lt_observables_noalloc: the lattice needs " + std::to_string(need) +
                                     " doubles of scratch, the fixed array holds " + std::to_string(NOALLOC_DOUBLES)};
    double* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(noalloc_mutex);
        if (ctx->device >= 0 && ctx->device < NOALLOC_MAX_DEVICES) base = noalloc_ptr[ctx->device];
    }
    if (!base) throw LtError{LT_ESTATE, "lt_observables_noalloc: no scratch address for this device"};
    const int nt = g.L[0];
    const int Vs = g.V / nt;
    const unsigned nchunk = nblocks(Vs, BS);
    double* part = base;
    double* fin = part + 9 * (size_t)nchunk * nt;
    double* out = fin + 3 * (size_t)nt;
    // every partial and every per-timeslice sum is written before it is read: nothing
    // has to start at zero
    hipLaunchKernelGGL(obs_kernel, dim3(3 * nchunk * nt), dim3(BS), 0, ctx->stream, (const double2*)u->d, g, Vs,
                       (int)nchunk, part);
    LT_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(obs_finish_kernel, dim3(nt), dim3(BS), 0, ctx->stream, (const double*)part, (int)nchunk, nt,
                       fin);
    LT_HIP_CHECK(hipGetLastError());
    hipLaunchKernelGGL(obs_final_kernel, dim3(1), dim3(64), 0, ctx->stream, (const double*)fin, nt, (double)g.V, out);
    LT_HIP_CHECK(hipGetLastError());
    LT_HIP_CHECK(hipMemcpyAsync(host_out, out, (4 + 2 * (size_t)nt) * sizeof(double), hipMemcpyDeviceToHost,
                                ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

void k_topcharge_density(lt_field u, double* host_q)
{
    lt_ctx ctx = u->ctx;
    const Geom& g = u->g;
    double* d = ctx->scratch_for((size_t)g.V);
    launch(ctx, "topcharge_density", qdensity_kernel, dim3(nblocks(g.V, BS)), dim3(BS), 0, (const double2*)u->d, g,
           d);
    LT_HIP_CHECK(hipMemcpyAsync(host_q, d, (size_t)g.V * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

}  // namespace lt
