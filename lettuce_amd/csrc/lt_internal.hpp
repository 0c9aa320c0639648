// lt_internal.hpp -- host-side objects behind the C ABI: contexts (device, stream,
// scratch, per-kernel event timing) and fields (device link buffer + Philox state),
// plus the launch helper every kernel goes through.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <exception>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "lettuce_hip.h"
#include "lt_device.hpp"

namespace lt {

void set_error(const std::string& msg);

struct LtError {
    int code;
    std::string msg;
};

#define LT_HIP_CHECK(expr)                                                                          \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess)                                                                       \
            throw ::lt::LtError{LT_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_)};        \
    } while (0)

// C ABI bodies: exceptions become a status code plus the lt_last_error message.
template <typename F>
int guarded(F&& f)
{
    try {
        return f();
    } catch (const LtError& e) {
        set_error(e.msg);
        return e.code;
    } catch (const std::exception& e) {
        set_error(e.what());
        return LT_ESTATE;
    }
}

inline int fail(int code, const std::string& msg)
{
    set_error(msg);
    return code;
}

struct ProfEntry {
    int launches = 0;
    double ms = 0.0;
};

}  // namespace lt

struct lt_ctx_s {
    int device = 0;
    hipStream_t stream = nullptr;
    int live = 0;              // fields, flows, CV workspaces and batches still holding this context
    // device scratch for reduction partials, grown on demand
    double* scratch = nullptr;
    size_t scratch_doubles = 0;
    // pinned host staging for reduction results
    double* host = nullptr;
    size_t host_doubles = 0;
    bool profiling = false;
    std::vector<std::pair<std::string, std::pair<hipEvent_t, hipEvent_t>>> pending;
    std::vector<std::pair<hipEvent_t, hipEvent_t>> event_pool;
    std::map<std::string, lt::ProfEntry> prof;

    // second link buffer of multi-level smearing, grown on demand and kept: allocating and
    // freeing 382 MB in every call took 6 to 9 ms where two stout levels of that field take 0.65 ms.
    // One buffer per context, of the largest field smeared so far; given back with the
    // context's last handle, and when another allocation of the library on this context fails
    // (all of them go through device_alloc).  A caller holds links_mutex while it enqueues the
    // launches that use the buffer (they are ordered by the stream), so threads sharing a context
    // do not interleave on it.
    std::mutex links_mutex;
    double2* links = nullptr;
    size_t links_n = 0;

    double* scratch_for(size_t n);
    double* host_for(size_t n);
    double2* links_for(size_t n);   // with links_mutex held
    void links_release();           // takes links_mutex
    void* device_alloc(size_t bytes);   // null when out of memory
    void handle_gone();             // a handle was destroyed (its stream work is done)
    void collect_profile();
};

namespace lt {
struct UpdateGraph;   // captured local-update loop body of a field (lt_update_sweeps)
}

struct lt_field_s {
    lt_ctx ctx = nullptr;
    lt::Geom g{};
    // thread -> site tiling of the per-parity link kernels, and of the plaquette pass, which
    // tuning the sweeps sets alone (the other kernels gain nothing from what suits that pass)
    lt::LinkMap map{}, plaq_map{};
    bool plaq_map_last = false;   // the tile set or tuned last is the plaquette pass's
    bool su3 = true;           // rows 0,1 stored, row 2 implied (false: general 3x3 matrices)
    bool view = false;         // d belongs to a replica batch (not freed, not swappable)
    double2* d = nullptr;      // 4 * 2 * 9 * Vh complex doubles
    uint64_t seed = 0;
    uint64_t counter = 0;
    lt::UpdateGraph* ug = nullptr;
    void set_map(const lt::LinkMap& m)
    {
        map = plaq_map = m;
        plaq_map_last = false;
    }
    const lt::LinkMap& last_map() const { return plaq_map_last ? plaq_map : map; }
    size_t bytes() const { return (size_t)72 * g.Vh * sizeof(double2); }
};

// MetaBiasPotential (LettuceGauge/actions/bias_potential/metadynamics.hpp:29-507)
struct lt_bias_s {
    std::vector<double> grid;
    double cv_current = 0.0, cv_min = 0.0, cv_max = 0.0, bin_width = 0.0, bin_width_inverse = 0.0;
    double weight = 0.0, width = 0.0, wt_param = 0.0, threshold = 0.0;
    int bins = 0;
    int well_tempered = 0;
    unsigned long long exceeded = 0;

    int bin_of(double cv) const { return (int)std::floor((cv - cv_min) * bin_width_inverse); }
    double cv_of(int i) const { return cv_min + i * bin_width; }
    // UpdatePotential (metadynamics.hpp:103-124)
    void deposit(double cv)
    {
        if (cv < cv_min || cv >= cv_max) exceeded += 1;
        const double wis = 1.0 / (width * width);
        for (size_t b = 0; b < grid.size(); ++b) {
            const double dist = cv - cv_of((int)b);
            if (well_tempered)
                grid[b] += weight * std::exp(-0.5 * wis * dist * dist - grid[b] / wt_param);
            else
                grid[b] += weight * std::exp(-0.5 * wis * dist * dist);
        }
    }
    // ReturnPotential (metadynamics.hpp:151-179)
    double potential(double cv) const
    {
        const int i = bin_of(cv);
        if ((unsigned)i < (unsigned)(bins)) {
            const double ic = (cv - cv_of(i)) * bin_width_inverse;
            return grid[i] * (1.0 - ic) + ic * grid[i + 1];
        }
        if (i < 0) {
            const double d = cv - cv_min;
            return grid.front() + threshold * d * d;
        }
        const double d = cv - cv_max;
        return grid.back() + threshold * d * d;
    }
    // ReturnDerivative (metadynamics.hpp:181-187)
    double derivative(double cv) const
    {
        const double h = 0.5 * bin_width;
        return bin_width_inverse * (potential(cv + h) - potential(cv - h));
    }
};

struct lt_flow_s {
    lt_field unflowed = nullptr;
    lt_field flowed = nullptr;
    int integrator = LT_FLOW_RK3;
    double eps = 0.0;
    double2* z = nullptr;      // RK3 Z field: su(3), 8 reals per link (ld_alg8 / st_alg8 layout)
    double2* tmp = nullptr;    // second link buffer for the Jacobi stages
};

namespace lt {

// Kernel launch with optional event timing on the context stream.
template <typename Kernel, typename... Args>
void launch(lt_ctx ctx, const char* name, Kernel kernel, dim3 grid, dim3 block, size_t shmem, Args... args)
{
    if (grid.x == 0 || grid.y == 0 || grid.z == 0) return;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    if (ctx->profiling) {
        if (!ctx->event_pool.empty()) {
            e0 = ctx->event_pool.back().first;
            e1 = ctx->event_pool.back().second;
            ctx->event_pool.pop_back();
        } else {
            LT_HIP_CHECK(hipEventCreate(&e0));
            LT_HIP_CHECK(hipEventCreate(&e1));
        }
        LT_HIP_CHECK(hipEventRecord(e0, ctx->stream));
    }
    hipLaunchKernelGGL(kernel, grid, block, shmem, ctx->stream, args...);
    LT_HIP_CHECK(hipGetLastError());
    if (ctx->profiling) {
        LT_HIP_CHECK(hipEventRecord(e1, ctx->stream));
        ctx->pending.push_back({name, {e0, e1}});
        if (ctx->pending.size() > 4096) ctx->collect_profile();
    }
}

inline unsigned nblocks(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }
// Map of a split colour launch over 1/colours of the sites.  tc, the timeslices that a chunk walks
// fastest, is the largest divisor of Nt up to Nt / 8 rounded up: one chunk for each XCD where Nt is
// a multiple of 8, elsewhere Nt / tc chunks, which the XCDs' ranges may cut (Nt = 28: 7 of 4, Nt = 20:
// 10 of 2).  Of 1 to 16 timeslices the best one is within 2 % of it.
inline SplitMap split_map(const Geom& g, int colours)
{
    int tc = 1;
    for (int d = 2; d <= (g.L[0] + 7) / 8; ++d)
        if (g.L[0] % d == 0) tc = d;
    SplitMap m;
    m.nt = g.V / g.L[0] / colours;
    m.dtc = make_div(tc);
    m.dper = make_div(tc * (int)nblocks(m.nt, SPLIT_LINKS));
    return m;
}
inline unsigned split_blocks(const Geom& g, const SplitMap& m) { return (unsigned)g.L[0] * nblocks(m.nt, SPLIT_LINKS); }
// grid size of a tiled link launch; refuses maps the kernels were not compiled for
inline unsigned map_blocks(const LinkMap& m)
{
    if (m.nthreads < 1 || m.nthreads > LT_LINK_BS || m.T[0] * m.T[1] * m.T[2] * m.T[3] != m.nthreads || m.tc < 1
        || m.N[0] % m.tc || m.yc < 1 || m.N[2] % m.yc)
        throw LtError{LT_ESTATE, "invalid thread-block tile for the link kernels"};
    return (unsigned)(m.N[0] * m.N[1] * m.N[2] * m.N[3]);
}
// block of the link launches that end in link_block_sum: the map's, in whole wavefronts
inline dim3 sum_block(const LinkMap& m) { return dim3((unsigned)(m.nthreads + 63) & ~63u); }

// The momentum / field update sequence of Integrators::HMC::{Leapfrog, OMF_2, OMF_4}
// (LettuceGauge/updates/hmc_gauge.hpp:48-75,155-190,241-295).  P(eps, sub) is a
// momentum update, sub marks the updates whose CV the MetaD path update samples.
void hmc_schedule(int kind, double tau, int n_step, const std::function<void(double, bool)>& P,
                  const std::function<void(double)>& U);
inline bool valid_integrator(int k)
{
    return k == LT_INT_LEAPFROG || k == LT_INT_OMF2 || k == LT_INT_OMF4 || k == LT_INT_LEAPFROG_SLOW ||
           k == LT_INT_OMF2_SLOW || k == LT_INT_OMF4_SLOW;
}

// Momentum kicks of a MetaD-HMC schedule: gauge force, bias force, or both in one update.
enum Kick { KICK_GAUGE = 1, KICK_BIAS = 2, KICK_BOTH = 3 };
// A KICK_BOTH momentum update P += a Algebra(st U^+) + bf F applied by the last kernel
// of the force computation instead of a separate pass over the stored force F.
struct MomentumKick {
    double2* P;
    double a, bf;
};
// Fields of a stout stack by level: level(j) is level j's field, tape(j) the exponent
// tape of the step from level j to level j + 1.
typedef std::function<const double2*(int)> LevelFn;
// The stout-force recursion (StoutForceRecursion, stout_smearing.hpp:122-234) from level
// hi down to level lo: the Lambda of level hi, then for k = hi..lo+1 the sigma update of
// level k, fused with the Lambda of level k-1 while k-1 > lo (the two Lambda buffers
// alternate); Sig holds the force as a matrix at both ends and is scratch between them.
// kick: applied by the update of
// level 1 instead of storing the level-0 force (lo == 0 only).  top_lambda_done: the
// Lambda of level hi is already in lam[0] (the clover derivative made it).
void k_stout_recursion_run(lt_ctx ctx, const Geom& g, const LinkMap& m, const LevelFn& level, const LevelFn& tape,
                           int hi, int lo, double2* Sig, double2* const lam[2], double rho,
                           const MomentumKick* kick = nullptr, bool top_lambda_done = false);
// The level below in a stout-force recursion step fused with its Lambda: its exponent tape
// and the Lambda buffer to write.
struct SigmaNext {
    const double2* T;
    double2* Lam;
};
// The MetaD-HMC sequence: the single-scale integrators kick with both forces
// (HMCMetaDKernel::UpdateMomenta, hmc_metadynamics.hpp:441-459); the multiple-timescale
// ones (hmc_metadynamics.hpp:28-238) kick the bias force on the outer scale and the
// gauge force on the inner OMF4.  P(eps, sub, kick); sub marks the path samples.
void metad_schedule(int kind, double tau, int n_step, const std::function<void(double, bool, int)>& P,
                    const std::function<void(double)>& U);
inline bool valid_metad_integrator(int k)
{
    return valid_integrator(k) || k == LT_INT_LEAPFROG_OMF4 || k == LT_INT_OMF2_OMF4_SLOW || k == LT_INT_OMF2_OMF4;
}

Geom make_geom(int nt, int nx, int ny, int nz);
// tile map with extents (tt, tx, ty, tz) over (t, x, y, z/2); returns false if they do not divide
bool make_linkmap(const Geom& g, int tt, int tx, int ty, int tz, LinkMap& m);
// Block of the clover derivative and of the stout-force recursion.  Their launches hold few
// waves per CU for long: with blocks of one wave a CU whose block is done gets the next one at
// once, with 128 threads it waits for both waves and the last blocks go on alone (recursion
// level 128 -> 64 threads: 16^4 90 -> 80 us, 16^3 x 32 157 -> 150, 24^4 374 -> 365, 32^4 1139 ->
// 1121, z = 48 252 -> 220 at 16^3 x 48; clover derivative -1 to -4 %, 12 x 8 x 10 x 14 34 -> 27;
// 256 threads: 24^4 380, 8^4 23.4 against 21.2).  The tape launches before them keep the default: two
// waves of a block share the links of their neighbours (32^4 526 -> 569 us with 64), except on
// small lattices (below).
constexpr int FORCE_BLOCK = 64;
// Lattices of up to this volume get blocks of one wave in every link kernel: their 4V links are at
// most one wave per SIMD, and blocks of two waves leave CUs empty while others hold two blocks.
// 128 -> 64 threads: four stout levels 8^4 32.0 -> 30.1 us, 10^4 53.1 -> 39.3, 12 x 8 x 10 x 14
// 57.6 -> 43.7, 16 x 8 x 8 x 16 57.1 -> 46.6; RK3 x 2 48.4 -> 45.6, 79.2 -> 60.8, 83.1 -> 65.5,
// 82.4 -> 68.5; an OMF2 trajectory of 8 steps 270 -> 260, 368 -> 310, 386 -> 334, 390 -> 347.  Beyond it nothing is left (12^4, 18 x 12 x 10 x 14 and 16^4
// within 2 % either way), and from 16^3 x 32 on the links that two waves share count (RK3 x 2
// 387 -> 407, 32^4 2980 -> 3121).
constexpr int SMALL_VOLUME = 16384;
// threads: block size, 0 for the default of the lattice's volume
LinkMap default_linkmap(const Geom& g, int threads = 0);
// same block shape and site order
inline bool same_map(const LinkMap& a, const LinkMap& b)
{
    for (int i = 0; i < 4; ++i)
        if (a.T[i] != b.T[i] || a.N[i] != b.N[i]) return false;
    return a.nthreads == b.nthreads && a.tc == b.tc && a.yc == b.yc && a.lin == b.lin && a.xr == b.xr;
}

// kernel launchers (defined in the .hip translation units)
void k_copy(lt_ctx ctx, const double2* src, double2* dst, size_t n);
// read-rate probe: nb blocks of 256 lanes, each reading iters 16-byte elements of buf
// (mask + 1 elements, a power of two) and writing one to out (nb * 256 elements)
void k_l2_read(lt_ctx ctx, const double2* buf, unsigned mask, int iters, double2* out, unsigned nb);
// y *= a over n complex entries (ReverseMomenta with a = -1)
void k_scale(lt_ctx ctx, double2* y, double a, size_t n);
void k_pack(lt_field f, const double* d_aos);
void k_unpack(lt_field f, double* d_aos);
void k_identity(lt_field f);
void k_haar(lt_field f, uint64_t seed);
void k_reunitarize(lt_field f);
void k_check(lt_field f, double* max_dev, long long* nonfinite);
void k_staple_field(lt_field u, lt_field out);
void k_or_sweep(lt_field u, int n, int schedule);
void k_hb_sweep(lt_field u, double beta, int n, int schedule);
// four-colour sweeps (lt_cb4.hip): the field's rows 0, 1 reordered in place between the
// plain cb order and the split order (to_split 1 / 0), and single colour launches that
// expect the split order
void k_cb_layout(lt_field u, int to_split);
void k_cb4_colour(lt_field u, bool heatbath, int mu, int colour, double prefactor, uint64_t counter, const char* name);
void k_cb4_colour_graph_hb(lt_field u, int mu, int colour, double prefactor, const uint64_t* state, int k);
void k_cb4_colour_action(lt_field u, bool heatbath, int mu, int colour, double prefactor, uint64_t counter,
                         double c_plaq, double c_rect, const char* name);
void k_cb4_plaq_partials(lt_field u, double* part);   // one partial per block of u->plaq_map's launch
// n_update x (n_hb heatbath + n_or overrelaxation sweeps) as one graph replayed per
// update, PlaquetteSum after each into plaq_host (may be null); and its teardown
void k_update_graph(lt_field u, double beta, int n_hb, int n_or, int schedule, int n_update, double* plaq_host);
void drop_update_graph(lt_field f);
// fused observables: per-timeslice plaquette sum, raw q, E_clov numerator -> host[3*Nt]
// BMW sites [n0, n0 + count) <-> big-endian file words (4 * K per site, K = 12 or
// 18), with per-block checksum partials (A, B) and, on unpacking, row-2 deviations
void k_bmw_pack(lt_field f, int K, long long n0, long long count, uint64_t* d_out, uint64_t* d_part);
void k_bmw_unpack(lt_field f, int K, long long n0, long long count, const uint64_t* d_in, uint64_t* d_part,
                  double* d_dev);
void k_parity(lt_field f, const double2* copy);
void k_staple_field_action(lt_field u, lt_field out, double c_plaq, double c_rect);
void k_or_sweep_action(lt_field u, int n, double c_plaq, double c_rect);
void k_heatbath_sweep_action(lt_field u, double beta, int n, double c_plaq, double c_rect);
void k_observables(lt_field u, double* host_out);
// sum over sites and planes of Re tr P, the planes of a site spread over its links (the HMC
// Hamiltonian keeps k_plaquette_sum, a plane pair per lane, which the replica batch repeats)
double k_plaquette_planes(lt_field u);
// its pass over the field alone: block sums into the context's scratch, whose number is returned
unsigned k_plaquette_partials(lt_field u);
// per-site clover charge density (V doubles, lexicographic order) into host memory
void k_topcharge_density(lt_field u, double* host_q);
// the fixed observables scratch of lt_observables_noalloc: its address on `device`
// (which must be current), looked up once per device
void noalloc_setup(int device);
// lt_observables' sums through the fixed scratch, final values computed on the device
void k_observables_noalloc(lt_field u, double* host_out);
void k_rect_sums(lt_field u, double out[2]);
double k_plaq_charge(lt_field u);
double k_wilson_loop(lt_field u, lt_field chain, int n0, int n1, int reset);
void k_polyakov_loop(lt_field u, double* re, double* im);
void k_stout(lt_ctx ctx, const Geom& g, const LinkMap& m, const double2* in, double2* out, double rho);
void k_flow_stage(lt_ctx ctx, const Geom& g, const LinkMap& m, const double2* in, double2* out, double2* z, double c_old,
                  double c_new, double c_exp, int read_z, int write_z);

}  // namespace lt
