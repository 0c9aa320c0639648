// lt_cb4.hip -- the four-colour (Checkerboard4) sweeps, iterators.hpp:141-169.
//
// A colour class of direction mu != z is every fourth z of a row, i.e. every other
// checkerboard index of one parity array.  In the plain cb order its loads and
// stores use half of every 128-byte line.  This translation unit is compiled with
// LT_SPLIT_CB = 1: its kernels address links in the order where every aligned group
// of 16 checkerboard indices holds its 8 even ones first (cbi in lt_device.hpp), in
// which a colour class reads and writes whole lines.  A four-colour sweep call
// reorders the field in place into that order (cb_layout_kernel), runs its colour
// launches and restores the plain order, so every other kernel of the library, all
// compiled with the plain order, sees the field as always.  The device code of each
// translation unit is its own code object; the inline device functions of the two
// orders never meet.
#define LT_SPLIT_CB 1
#include "lt_internal.hpp"
#include "lt_bodies.hpp"
#include "lt_sweep.hpp"

namespace lt {

namespace {

constexpr int RBS = 256;

// Colours 1 and 3 walk the blocks backwards (xcd_block_dir): consecutive colour launches then
// start where the previous one ended.  In a captured update the Philox counter is state[0] + k
// from device memory.
// Wilson staple, between events, against one lane per link: overrelaxation 8^4 12.1 -> 8.3 us,
// 16^4 12.7 -> 9.2, 28^4 76 -> 51.8, 32^4 77.3 -> 75.2; heatbath 8^4 21.7 -> 11.7, 16^4 21.3 ->
// 13.5, 28^4 89 -> 63.3, 32^4 89 -> 80.  Small ones are bound by the latency of one link, large
// ones by the memory behind the L2.
// Rectangle staple: one lane per link with the sum parked in LDS ran about 9500 FP64
// instructions in a row at two waves per SIMD, 186 us per overrelaxation launch at 24^4 and 322
// us at 32^4; now 81.6 and 199 us (heatbath 195 -> 92 us at 24^4: three wavefronts per SIMD with 22
// registers, 60 bytes a lane, spilled; two without spills are no faster).  About half of its lines miss
// the L2: 385 MB a launch at 24^4, 53 us at the rate at which the memory-side cache reads.
template <bool HEATBATH, int KIND, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(split_eu(HEATBATH, KIND, WAVES))))
sweep_cb4_kernel(double2* __restrict__ U, Geom g, int mu, int colour, double prefactor, uint64_t seed, uint64_t counter,
                 const uint64_t* __restrict__ state, int k, double c_plaq, double c_rect, SplitMap map)
{
    __shared__ SplitShared<HEATBATH, WAVES> sh;
    if (HEATBATH && state) counter = state[0] + (uint64_t)k;
    int c[4], s = 0;
    const int i = split_index(map, xcd_block_dir(blockIdx.x, gridDim.x, colour & 1));
    const bool on = i >= 0 && cb4_site(g, mu, colour, i, c, s);
    update_links_split<HEATBATH, KIND, WAVES>(U, g, mu, on, s, c, prefactor, seed, counter, c_plaq, c_rect, sh);
}

// PlaquetteSum block partials of a captured four-colour update (the field is in the
// split order inside the graph); the same terms, launch and partials as the
// plain-order kernel
__global__ void LT_LINK_KERNEL cb4_plaq_kernel(const double2* __restrict__ U, Geom g, LinkMap m, double* part)
{
    plaq_link_partials(U, g, m, part);
}

// In-place reorder of rows 0 and 1 of every link between the plain cb order and the
// split order.  One lane per slot of a group of 16 (a group lies in one wavefront):
// each lane loads its slot, the wavefront's loads complete before its stores, and no
// other wavefront touches the group.  A last group of 8 (Vh not a multiple of 16)
// keeps its order in both layouts.
__global__ void __launch_bounds__(RBS) cb_layout_kernel(double2* __restrict__ U, Geom g, int to_split)
{
    const long long vh16 = g.Vh & ~15;
    const long long id = (long long)blockIdx.x * RBS + threadIdx.x;
    if (id >= 48 * vh16) return;
    const int a = (int)(id / vh16);            // (mu*2 + parity)*6 + component
    const int e = (int)(id - a * vh16);
    const int grp = e & ~15, l = e & 15;
    const int dst = to_split ? ((l & 1) << 3) | (l >> 1)    // cb l -> slot
                             : (l < 8 ? 2 * l : 2 * (l - 8) + 1);   // slot l -> cb
    double2* p = U + (size_t)(a % 6) * slot_stride(g);
    const double2 v = p[slot_base(g, a / 6, 9, grp + l)];
    p[slot_base(g, a / 6, 9, grp + dst)] = v;
}

}  // namespace

void k_cb_layout(lt_field u, int to_split)
{
    if (!u->su3) throw LtError{LT_EINVAL, "four-colour sweeps need an SU(3) gauge field"};
    const long long n = 48LL * (u->g.Vh & ~15);
    if (n) launch(u->ctx, "cb_layout", cb_layout_kernel, dim3(nblocks(n, RBS)), dim3(RBS), 0, u->d, u->g, to_split);
}

namespace {

template <bool HEATBATH, int KIND, int WAVES>
void colour_waves(lt_field u, const char* name, int mu, int colour, double prefactor, uint64_t counter,
                  const uint64_t* state, int k, double c_plaq, double c_rect)
{
    const SplitMap m = split_map(u->g, 4);
    launch(u->ctx, name, sweep_cb4_kernel<HEATBATH, KIND, WAVES>, dim3(split_blocks(u->g, m)), dim3(64 * WAVES), 0, u->d,
           u->g, mu, colour, prefactor, u->seed, counter, state, k, c_plaq, c_rect, m);
}

// Wavefronts per block.  Three, of which four blocks fit a compute unit, wherever the parts are
// of one wavefront's size: the heatbath (20^4 24.8 -> 22.6 us, 24^4 37.8 -> 37.2 against six).
// Overrelaxation takes three where rows of a multiple of 32 z give a class whole 128-byte lines
// per row (32^4 75.2 against 79.8 us with six, 16^2 x 32^2 20.8 and 21.6) and six where rows
// leave half lines, which the six wavefronts of a block then share in the L1 (24^4 30.0 us
// against 34.0 with three, 28^4 51.8 and 59.7, 48 x 24^3 51 and 62).  The rectangle staple's
// parts spill with two sides in a wavefront.
template <bool HEATBATH, int KIND>
void colour_launch(lt_field u, const char* name, int mu, int colour, double prefactor, uint64_t counter,
                   const uint64_t* state, int k, double c_plaq, double c_rect)
{
    if constexpr (KIND == SPLIT_RECT)
        colour_waves<HEATBATH, KIND, 6>(u, name, mu, colour, prefactor, counter, state, k, c_plaq, c_rect);
    else if (HEATBATH || u->g.L[3] % 32 == 0)
        colour_waves<HEATBATH, KIND, 3>(u, name, mu, colour, prefactor, counter, state, k, c_plaq, c_rect);
    else
        colour_waves<false, KIND, 6>(u, name, mu, colour, prefactor, counter, state, k, c_plaq, c_rect);
}

}  // namespace

void k_cb4_colour(lt_field u, bool heatbath, int mu, int colour, double prefactor, uint64_t counter, const char* name)
{
    auto* f = heatbath ? colour_launch<true, SPLIT_WILSON> : colour_launch<false, SPLIT_WILSON>;
    f(u, name, mu, colour, prefactor, counter, nullptr, 0, 1.0, 0.0);
}

void k_cb4_colour_graph_hb(lt_field u, int mu, int colour, double prefactor, const uint64_t* state, int k)
{
    colour_launch<true, SPLIT_WILSON>(u, "hb_cb4", mu, colour, prefactor, 0, state, k, 1.0, 0.0);
}

void k_cb4_colour_action(lt_field u, bool heatbath, int mu, int colour, double prefactor, uint64_t counter,
                         double c_plaq, double c_rect, const char* name)
{
    auto* f = heatbath ? (c_rect != 0.0 ? colour_launch<true, SPLIT_RECT> : colour_launch<true, SPLIT_SCALED>)
                       : (c_rect != 0.0 ? colour_launch<false, SPLIT_RECT> : colour_launch<false, SPLIT_SCALED>);
    f(u, name, mu, colour, prefactor, counter, nullptr, 0, c_plaq, c_rect);
}

void k_cb4_plaq_partials(lt_field u, double* part)
{
    launch(u->ctx, "plaquette", cb4_plaq_kernel, dim3(8 * map_blocks(u->plaq_map)), sum_block(u->plaq_map), 0,
           (const double2*)u->d, u->g, u->plaq_map, part);
}

}  // namespace lt
