// lt_hmc.hip -- HMC building blocks: Gaussian su(3) momenta from Philox, the gauge
// (and metadynamics) momentum update, the exponential field update and the
// deterministic reductions of the Hamiltonian (plaquette sum, kinetic energy).
//
// Forces are general 3x3 fields (all 9 entries stored), momenta too unless alg says that they
// are in 8 reals (lt_bodies.hpp).  The per-link bodies live in lt_bodies.hpp and are shared
// with the replica-batched kernels.
#include "lt_internal.hpp"
#include "lt_bodies.hpp"

namespace lt {

namespace {

constexpr int RBS = 256;   // reduction block size

template <bool ALG>
__global__ void LT_LINK_KERNEL momentum_kernel(double2* __restrict__ P, Geom g, LinkMap m, uint64_t seed,
                                               uint64_t counter)
{
    body_momentum<ALG>(P, g, m, link_block(m, blockIdx.x, gridDim.x), seed, counter);
}

// 16^3 x 32: 54.5 us with momenta in 8 reals, 60 as whole matrices; bound by VALU issue and
// latency at the two waves per SIMD of the pipelined staple.
template <bool ALG>
__global__ void LT_LINK_KERNEL force_update_kernel(const double2* __restrict__ U, double2* __restrict__ P,
                                                   const double2* __restrict__ F, Geom g, LinkMap m, double a, double b)
{
    body_force_update<ALG>(U, P, F, g, m, link_block(m, blockIdx.x, gridDim.x), a, b);
}

// Memory bound: 16^3 x 32 22.9 us with momenta in 8 reals (5.9 TB/s), 28.9 as whole matrices.
template <bool ALG>
__global__ void LT_LINK_KERNEL field_update_kernel(double2* __restrict__ U, const double2* __restrict__ P, Geom g,
                                                   LinkMap m, double eps)
{
    body_field_update<ALG>(U, P, g, m, link_block(m, blockIdx.x, gridDim.x), eps);
}

__device__ __forceinline__ void block_sum(double v, double* out)
{
    block_sum_to<RBS>(v, out);
}

// block b (XCD-remapped) takes plane pair b % 3 of site chunk b / 3 (one lane per site with all
// six planes needs a whole SIMD per wave: 16^3 x 32 29 -> 20 us between events)
__global__ void __launch_bounds__(RBS) plaq_kernel(const double2* __restrict__ U, Geom g, double* part)
{
    const int b = xcd_block(blockIdx.x, gridDim.x);
    block_sum(body_plaq_pair(U, g, (b / 3) * RBS + threadIdx.x, b % 3), part + b);
}

template <bool ALG>
__global__ void __launch_bounds__(RBS) kinetic_kernel(const double2* __restrict__ P, Geom g, double* part)
{
    const int i = blockIdx.x * RBS + threadIdx.x;
    block_sum(i < 8 * g.Vh ? body_kinetic_link<ALG>(P, g, i) : 0.0, part + blockIdx.x);
}

template <bool WHOLE>
__global__ void __launch_bounds__(RBS) momentum_entry_kernel(double2* __restrict__ P, const double2* __restrict__ F, Geom g,
                                                             double a)
{
    const int i = blockIdx.x * RBS + threadIdx.x;
    if (i < 8 * g.Vh) body_momentum_entry<WHOLE>(P, F, g, i, a);
}

// single block: ordered sum of n partials
__global__ void __launch_bounds__(RBS) finish_kernel(const double* part, int n, double* out)
{
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += RBS) acc += part[i];
    block_sum(acc, out);
}

double reduce(lt_ctx ctx, unsigned nb, double* part, double* fin)
{
    launch(ctx, "reduce_finish", finish_kernel, dim3(1), dim3(RBS), 0, (const double*)part, (int)nb, fin);
    double* h = ctx->host_for(1);
    LT_HIP_CHECK(hipMemcpyAsync(h, fin, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return h[0];
}

}  // namespace

void k_random_momentum(lt_field P, uint64_t seed, uint64_t counter, bool alg)
{
    const LinkMap& m = P->map;
    auto* k = alg ? momentum_kernel<true> : momentum_kernel<false>;
    launch(P->ctx, "momentum", k, dim3(8 * map_blocks(m)), dim3(m.nthreads), 0, P->d, P->g, m, seed,
           counter);
}

void k_force_update(lt_field U, lt_field P, const double2* F, double a, double b, bool alg)
{
    const LinkMap& m = U->map;
    auto* k = alg ? force_update_kernel<true> : force_update_kernel<false>;
    launch(U->ctx, "force_update", k, dim3(8 * map_blocks(m)), dim3(m.nthreads), 0,
           (const double2*)U->d, P->d, F, U->g, m, a, b);
}

void k_field_update(lt_field U, lt_field P, double eps, bool alg)
{
    const LinkMap& m = U->map;
    auto* k = alg ? field_update_kernel<true> : field_update_kernel<false>;
    launch(U->ctx, "field_update", k, dim3(8 * map_blocks(m)), dim3(m.nthreads), 0, U->d,
           (const double2*)P->d, U->g, m, eps);
}

double k_plaquette_sum(lt_field U)
{
    lt_ctx ctx = U->ctx;
    const unsigned nb = 3 * nblocks(U->g.V, RBS);
    double* part = ctx->scratch_for(nb + 1);
    launch(ctx, "plaquette", plaq_kernel, dim3(nb), dim3(RBS), 0, (const double2*)U->d, U->g, part);
    return reduce(ctx, nb, part, part + nb);
}

double k_kinetic(lt_field P, bool alg)
{
    lt_ctx ctx = P->ctx;
    unsigned nb = nblocks(4LL * P->g.V, RBS);
    double* part = ctx->scratch_for(nb + 1);
    auto* k = alg ? kinetic_kernel<true> : kinetic_kernel<false>;
    launch(ctx, "kinetic", k, dim3(nb), dim3(RBS), 0, (const double2*)P->d, P->g, part);
    return reduce(ctx, nb, part, part + nb);
}

// momenta in 8 reals: P += a F, and P as whole matrices
void k_momentum_kick(lt_ctx ctx, const Geom& g, double2* P, const double2* F, double a)
{
    launch(ctx, "momentum_kick", momentum_entry_kernel<false>, dim3(nblocks(8LL * g.Vh, RBS)), dim3(RBS), 0, P, F, g, a);
}
void k_momentum_whole(lt_field P)
{
    launch(P->ctx, "momentum_whole", momentum_entry_kernel<true>, dim3(nblocks(8LL * P->g.Vh, RBS)), dim3(RBS), 0, P->d,
           (const double2*)nullptr, P->g, 0.0);
}

}  // namespace lt
