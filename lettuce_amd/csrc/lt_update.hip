// lt_update.hip -- checkerboarded local updates: Wilson staple, SU(2)-subgroup
// overrelaxation and Cabibbo-Marinari pseudo-heatbath with Philox draws.
//
// One launch updates one colour class of one direction mu.  With the 2-colour
// schedule a colour class is exactly one parity array, and every link is written in
// place by one lane; the staple only reads links of other directions or of the opposite
// parity, so the update is race free.  The 4-colour schedule (colour (sum + x_mu) mod 4)
// runs in lt_cb4.hip on the field reordered for the duration of the call.
#include "lt_internal.hpp"
#include "lt_bodies.hpp"
#include "lt_sweep.hpp"

namespace lt {

namespace {

constexpr int BS = LT_LINK_BS;

// Three wavefronts per 64 links (update_links_split).  Every launch of a sweep reads all eight
// half-fields, so the parity-1 launch of each direction walks the blocks backwards
// (xcd_block_dir) and starts on the lines the parity-0 launch touched last, which are still in
// the L2 and the memory-side cache.  In a captured update the Philox counter is read from
// device memory (state[0], advanced by the graph itself) instead of a launch argument, so one
// captured graph serves every replay; sweep k of an update draws with counter state[0] + k, as
// the eager sweeps draw with the field's counter.
// Small launches are bound by the latency of one link (8^4: 7.7 us between events, heatbath
// 11.5, of which about 6 us are the launch itself), large ones by the memory behind the L2
// (32^4: 94 us for 453 MB).  Overrelaxation and heatbath with one lane per link: 16^4 10.9 and
// 21 us, now 10.0 and 16; 24^4 36 and 57, now 32 and 45; 28^4 82 and 98, now 54 and 71; 32^4
// 96.7 and 126, now 94 and 114.  Only where the blocks of three just pass one round of the
// GPU's 1024 or two is one lane as good (20^4: 25.0 against 26.1 us; the heatbath there 37.4
// and 29.8).
constexpr int CB2_WAVES = 3;
template <bool HEATBATH>
__global__ void __launch_bounds__(64 * CB2_WAVES)
__attribute__((amdgpu_waves_per_eu(split_eu(HEATBATH, SPLIT_WILSON, CB2_WAVES))))
sweep_cb2_kernel(double2* __restrict__ U, Geom g, int mu, int par, double prefactor, uint64_t seed, uint64_t counter,
                 const uint64_t* __restrict__ state, int k, SplitMap map)
{
    __shared__ SplitShared<HEATBATH, CB2_WAVES> sh;
    if (HEATBATH && state) counter = state[0] + (uint64_t)k;
    int c[4] = {0, 0, 0, 0}, s = 0;
    const int i = split_index(map, xcd_block_dir(blockIdx.x, gridDim.x, par));
    if (i >= 0) s = site_of_cb(g, i, par, c);
    update_links_split<HEATBATH, SPLIT_WILSON, CB2_WAVES>(U, g, mu, i >= 0, s, c, prefactor, seed, counter, 1.0, 0.0, sh);
}

// PlaquetteSum of the captured update: per-block sums (the block tree of the HMC
// reductions), then one ordered sum written to plaq[state[1]]
constexpr int RBS = 256;
__device__ __forceinline__ void block_sum1(double v, double* out)
{
    block_sum_to<RBS>(v, out);
}
// plaquette sum over the field's link map, one partial per block
__global__ void LT_LINK_KERNEL upd_plaq_kernel(const double2* __restrict__ U, Geom g, LinkMap m, double* part)
{
    plaq_link_partials(U, g, m, part);
}
unsigned plaq_parts(const LinkMap& m) { return 8u * map_blocks(m); }
__global__ void __launch_bounds__(RBS) plaq_sum_kernel(const double* __restrict__ part, int n, double* out)
{
    block_sum1(partials_sum<RBS>(part, n), out);
}
// the same sum into the plaquette slot of a captured update
__global__ void __launch_bounds__(RBS) upd_plaq_finish_kernel(const double* __restrict__ part, int n,
                                                              const uint64_t* __restrict__ state, double* plaq)
{
    block_sum1(partials_sum<RBS>(part, n), plaq + state[1]);
}
// end of a captured update: the next one draws n_hb counters later and writes the next slot
__global__ void upd_advance_kernel(uint64_t* state, int n_hb)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        state[0] += (uint64_t)n_hb;
        state[1] += 1;
    }
}

template <bool RECT>
__global__ void __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(2)))
staple_action_kernel(const double2* __restrict__ U, double2* __restrict__ out, Geom g, double c_plaq, double c_rect)
{
    const long long id = (long long)blockIdx.x * BS + threadIdx.x;
    if (id >= 4LL * g.V) return;
    const int s = (int)(id >> 2), mu = (int)(id & 3);
    int c[4];
    coords_of(g, s, c);
    const int par = parity_of(c);
    st_link(out, g, s, mu, par, staple_action<RECT>(U, g, s, c, mu, par, c_plaq, c_rect));
}

__global__ void LT_LINK_KERNEL staple_field_kernel(const double2* __restrict__ U, double2* __restrict__ out, Geom g,
                                                   LinkMap m)
{
    int mu = blockIdx.y >> 1, par = blockIdx.y & 1;
    int c[4], s;
    if (!map_site(g, m, par, c, s)) return;
    st_link(out, g, s, mu, par, staple(U, g, s, c, mu));
}

template <bool HEATBATH>
void cb2_colour(lt_field u, const char* name, int mu, int par, double prefactor, uint64_t counter, const uint64_t* state,
               int k)
{
    const SplitMap m = split_map(u->g, 2);
    launch(u->ctx, name, sweep_cb2_kernel<HEATBATH>, dim3(split_blocks(u->g, m)), dim3(64 * CB2_WAVES),
           0, u->d, u->g, mu, par, prefactor, u->seed, counter, state, k, m);
}

// n sweeps; the four-colour ones (split) expect the field in the split order
template <bool HEATBATH>
void sweep_launches(lt_field u, int n, int schedule, double prefactor, const char* name)
{
    for (int k = 0; k < n; ++k) {
        uint64_t counter = HEATBATH ? u->counter++ : 0;
        for (int mu = 0; mu < 4; ++mu) {
            if (schedule == LT_CB4) {
                for (int col = 0; col < 4; ++col) k_cb4_colour(u, HEATBATH, mu, col, prefactor, counter, name);
            } else {
                for (int par = 0; par < 2; ++par) cb2_colour<HEATBATH>(u, name, mu, par, prefactor, counter, nullptr, 0);
            }
        }
    }
}

template <bool HEATBATH>
void sweeps(lt_field u, int n, int schedule, double prefactor, const char* name)
{
    if (schedule == LT_CB4 && n > 0) {
        k_cb_layout(u, 1);
        sweep_launches<HEATBATH>(u, n, schedule, prefactor, name);
        k_cb_layout(u, 0);
    } else {
        sweep_launches<HEATBATH>(u, n, schedule, prefactor, name);
    }
}

template <bool HEATBATH>
void sweeps_action(lt_field u, int n, double prefactor, double c_plaq, double c_rect, const char* name)
{
    if (n <= 0) return;
    k_cb_layout(u, 1);
    for (int k = 0; k < n; ++k) {
        uint64_t counter = HEATBATH ? u->counter++ : 0;
        for (int mu = 0; mu < 4; ++mu)
            for (int col = 0; col < 4; ++col) k_cb4_colour_action(u, HEATBATH, mu, col, prefactor, counter, c_plaq, c_rect, name);
    }
    k_cb_layout(u, 0);
}

}  // namespace

void k_staple_field_action(lt_field u, lt_field out, double c_plaq, double c_rect)
{
    auto* k = c_rect != 0.0 ? staple_action_kernel<true> : staple_action_kernel<false>;
    launch(u->ctx, "staple_action", k, dim3(nblocks(4LL * u->g.V, BS)), dim3(BS), 0, (const double2*)u->d, out->d, u->g,
           c_plaq, c_rect);
}

void k_or_sweep_action(lt_field u, int n, double c_plaq, double c_rect)
{
    sweeps_action<false>(u, n, 0.0, c_plaq, c_rect, "or_action");
}

void k_heatbath_sweep_action(lt_field u, double beta, int n, double c_plaq, double c_rect)
{
    sweeps_action<true>(u, n, 3.0 / beta, c_plaq, c_rect, "hb_action");
}

void k_staple_field(lt_field u, lt_field out)
{
    const LinkMap& m = u->map;
    launch(u->ctx, "staple_field", staple_field_kernel, dim3(map_blocks(m), 8), dim3(m.nthreads), 0,
           (const double2*)u->d, out->d, u->g, m);
}

// ---- the local-update loop body as one replayed graph --------------------------
struct UpdateGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    // what the captured launches depend on
    const double2* d = nullptr;
    LinkMap m{};
    uint64_t seed = 0;
    double beta = 0.0;
    int n_hb = -1, n_or = -1, schedule = 0, with_plaq = 0;
    // device memory: state[0] = Philox counter, state[1] = plaquette slot; partials; plaquette sums
    uint64_t* state = nullptr;
    double* part = nullptr;
    double* plaq = nullptr;
    size_t cap = 0;        // plaquette sums held by plaq
    unsigned part_cap = 0;  // partials held by part
    unsigned nb = 0;        // partials of the present launch map

    void drop_exec()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }
    ~UpdateGraph()
    {
        drop_exec();
        if (state) (void)hipFree(state);
        if (part) (void)hipFree(part);
        if (plaq) (void)hipFree(plaq);
    }
};

void drop_update_graph(lt_field f)
{
    delete f->ug;
    f->ug = nullptr;
}

namespace {

// the launches of one update, in the order of the eager sweeps
void enqueue_update(lt_field u, UpdateGraph& G, double prefactor)
{
    lt_ctx ctx = u->ctx;
    for (int k = 0; k < G.n_hb; ++k)
        for (int mu = 0; mu < 4; ++mu) {
            if (G.schedule == LT_CB4) {
                for (int col = 0; col < 4; ++col) k_cb4_colour_graph_hb(u, mu, col, prefactor, G.state, k);
            } else {
                for (int par = 0; par < 2; ++par) cb2_colour<true>(u, "hb_cb2", mu, par, prefactor, 0, G.state, k);
            }
        }
    sweep_launches<false>(u, G.n_or, G.schedule, 0.0, G.schedule == LT_CB4 ? "or_cb4" : "or_cb2");
    if (G.with_plaq) {
        if (G.schedule == LT_CB4)
            k_cb4_plaq_partials(u, G.part);
        else
            launch(ctx, "plaquette", upd_plaq_kernel, dim3(8 * map_blocks(u->plaq_map)), sum_block(u->plaq_map), 0,
                   (const double2*)u->d, u->g, u->plaq_map, G.part);
        launch(ctx, "reduce_finish", upd_plaq_finish_kernel, dim3(1), dim3(RBS), 0, (const double*)G.part, (int)G.nb,
               (const uint64_t*)G.state, G.plaq);
    }
    launch(ctx, "update_advance", upd_advance_kernel, dim3(1), dim3(64), 0, G.state, G.n_hb);
}

}  // namespace

void k_update_graph(lt_field u, double beta, int n_hb, int n_or, int schedule, int n_update, double* plaq_host)
{
    lt_ctx ctx = u->ctx;
    if (!u->ug) u->ug = new UpdateGraph();
    UpdateGraph& G = *u->ug;
    const int with_plaq = plaq_host ? 1 : 0;
    auto alloc = [&](size_t bytes) {
        void* p = ctx->device_alloc(bytes);
        if (!p) throw LtError{LT_ENOMEM, "update graph allocation failed"};
        return p;
    };
    if (!G.state) G.state = (uint64_t*)alloc(2 * sizeof(uint64_t));
    // plaquette partials: one per block of the pass's present map
    const unsigned np = plaq_parts(u->plaq_map);
    if (np > G.part_cap) {
        G.drop_exec();
        if (G.part) LT_HIP_CHECK(hipFree(G.part));
        G.part = nullptr;
        G.part_cap = 0;
        G.part = (double*)alloc((size_t)np * sizeof(double));
        G.part_cap = np;
    }
    G.nb = np;
    if (with_plaq && (size_t)n_update > G.cap) {
        G.drop_exec();
        if (G.plaq) LT_HIP_CHECK(hipFree(G.plaq));
        G.plaq = nullptr;
        G.cap = 0;
        G.plaq = (double*)alloc((size_t)n_update * sizeof(double));
        G.cap = (size_t)n_update;
    }
    if (!G.exec || G.d != u->d || !same_map(G.m, u->plaq_map) || G.seed != u->seed || G.beta != beta || G.n_hb != n_hb ||
        G.n_or != n_or || G.schedule != schedule || G.with_plaq != with_plaq) {
        G.drop_exec();
        G.d = u->d;
        G.m = u->plaq_map;
        G.seed = u->seed;
        G.beta = beta;
        G.n_hb = n_hb;
        G.n_or = n_or;
        G.schedule = schedule;
        G.with_plaq = with_plaq;
        const bool prof = ctx->profiling;
        ctx->profiling = false;
        LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
        LT_HIP_CHECK(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
        try {
            enqueue_update(u, G, 3.0 / beta);
        } catch (...) {
            hipGraph_t gr = nullptr;
            (void)hipStreamEndCapture(ctx->stream, &gr);
            if (gr) (void)hipGraphDestroy(gr);
            ctx->profiling = prof;
            throw;
        }
        ctx->profiling = prof;
        LT_HIP_CHECK(hipStreamEndCapture(ctx->stream, &G.graph));
        LT_HIP_CHECK(hipGraphInstantiate(&G.exec, G.graph, nullptr, nullptr, 0));
    }
    const uint64_t st[2] = {u->counter, 0};
    LT_HIP_CHECK(hipMemcpyAsync(G.state, st, sizeof(st), hipMemcpyHostToDevice, ctx->stream));
    // a four-colour graph runs on the split order (its kernels are lt_cb4.hip's)
    if (schedule == LT_CB4) k_cb_layout(u, 1);
    for (int i = 0; i < n_update; ++i) LT_HIP_CHECK(hipGraphLaunch(G.exec, ctx->stream));
    if (schedule == LT_CB4) k_cb_layout(u, 0);
    u->counter += (uint64_t)n_hb * (uint64_t)n_update;
    if (plaq_host)
        LT_HIP_CHECK(hipMemcpyAsync(plaq_host, G.plaq, (size_t)n_update * sizeof(double), hipMemcpyDeviceToHost,
                                    ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
}

unsigned k_plaquette_partials(lt_field u)
{
    const unsigned nb = plaq_parts(u->plaq_map);
    launch(u->ctx, "plaquette", upd_plaq_kernel, dim3(nb), sum_block(u->plaq_map), 0, (const double2*)u->d, u->g,
           u->plaq_map, u->ctx->scratch_for((size_t)nb + 1));
    return nb;
}

double k_plaquette_planes(lt_field u)
{
    lt_ctx ctx = u->ctx;
    const unsigned nb = k_plaquette_partials(u);
    double* part = ctx->scratch;
    launch(ctx, "plaquette_sum", plaq_sum_kernel, dim3(1), dim3(RBS), 0, (const double*)part, (int)nb, part + nb);
    double* h = ctx->host_for(1);
    LT_HIP_CHECK(hipMemcpyAsync(h, part + nb, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    LT_HIP_CHECK(hipStreamSynchronize(ctx->stream));
    return h[0];
}

void k_or_sweep(lt_field u, int n, int schedule)
{
    sweeps<false>(u, n, schedule, 0.0, schedule == LT_CB4 ? "or_cb4" : "or_cb2");
}

void k_hb_sweep(lt_field u, double beta, int n, int schedule)
{
    sweeps<true>(u, n, schedule, 3.0 / beta, schedule == LT_CB4 ? "hb_cb4" : "hb_cb2");
}

}  // namespace lt
