// The collide launches of the handle API, by boundary, force and LES.  Each
// storage type has a source of its own that instantiates launch_step
// (launch_*.hip), so that they compile side by side.
#pragma once

#include "engine_internal.hpp"

using namespace bgk;
using namespace bgk::eng;

namespace {

template <typename S, int BX, int BY, int BZ, bool OB, int FM, int SR>
void launch_fused(bgk_handle& h, bool pair)
{
    const FusedArgs<S> p = fused_args<S>(h, h.cur, h.rest);
    if constexpr (kPairs<S>) {
        if (pair) {
            // obstacle forms always stream: they take the longest to compile,
            // and a plain-store copy of each would double that
            if constexpr (!OB) {
                if (keep_in_cache(lattice_bytes(h))) {
                    launch_pair<S, BX, BY, BZ, OB, FM, false>(p, h.pgrid, h.stream);
                    return;
                }
            }
            launch_pair<S, BX, BY, BZ, OB, FM, true>(p, h.pgrid, h.stream);
            return;
        }
    }
    if (h.compact) {
        hipLaunchKernelGGL((collide_compact<S, BX, BY, BZ, OB, FM, SR>),
                           dim3((unsigned)ceil_div(p.lend, 256), (unsigned)p.n), dim3(256), compact_lds_cap<S>(),
                           h.stream, p);
        return;
    }
    const RowMap rm = row_map(p.l);
    if constexpr (sizeof(S) == 2) {
        if (p.lend <= p.l) {
            hipLaunchKernelGGL((collide_fused<S, BX, BY, BZ, OB, FM, SR, false>), fused_grid(rm, p.m, p.n),
                               fused_block(rm), 0, h.stream, p, rm);
            return;
        }
    }
    hipLaunchKernelGGL((collide_fused<S, BX, BY, BZ, OB, FM, SR>), fused_grid(rm, p.m, p.n), fused_block(rm), 0,
                       h.stream, p, rm);
}

// L = 4 selects the Smagorinsky LES relaxation (FMODE bit 2)
template <typename S, int SR, int L>
void dispatch_fused_les(bgk_handle& h, bool pair)
{
    const bgk_config& c = h.cfg;
    switch (c.boundary) {
        case BGK_BC_DRIVEN: launch_fused<S, AX_WALL, AX_WALL, AX_LID, false, L, SR>(h, pair); break;
        case BGK_BC_PERIODIC:
            if (h.has_obs)
                launch_fused<S, AX_PERIODIC, AX_PERIODIC, AX_PERIODIC, true, L, SR>(h, pair);
            else
                launch_fused<S, AX_PERIODIC, AX_PERIODIC, AX_PERIODIC, false, L, SR>(h, pair);
            break;
        case BGK_BC_CHANNEL:
            if (c.wall_axis == 2) {  // walls at y = 1, m; x and z periodic
                if (c.force_axis == 3)
                    launch_fused<S, AX_PERIODIC, AX_WALL, AX_PERIODIC, false, 3 | L, SR>(h, pair);
                else
                    launch_fused<S, AX_PERIODIC, AX_WALL, AX_PERIODIC, false, 1 | L, SR>(h, pair);
            } else if (c.force_axis == 2) {
                launch_fused<S, AX_PERIODIC, AX_PERIODIC, AX_WALL, false, 2 | L, SR>(h, pair);
            } else if (c.force_axis == 3) {
                launch_fused<S, AX_PERIODIC, AX_PERIODIC, AX_WALL, false, 3 | L, SR>(h, pair);
            } else {
                launch_fused<S, AX_PERIODIC, AX_PERIODIC, AX_WALL, false, 1 | L, SR>(h, pair);
            }
            break;
        default:
            if (h.has_obs)
                launch_fused<S, AX_HALO, AX_PERIODIC, AX_PERIODIC, true, L, SR>(h, pair);
            else
                launch_fused<S, AX_HALO, AX_PERIODIC, AX_PERIODIC, false, L, SR>(h, pair);
            break;
    }
}

template <typename S, int SR>
void dispatch_fused(bgk_handle& h, bool pair)
{
    if (h.cfg.les)
        dispatch_fused_les<S, SR, 4>(h, pair);
    else
        dispatch_fused_les<S, SR, 0>(h, pair);
}

}  // namespace

namespace bgk {
namespace eng {

template <typename S>
void launch_step(bgk_handle& h, bool pair)
{
    if constexpr (sizeof(S) == 2) {
        if (h.cfg.rounding) {
            dispatch_fused<S, 1>(h, pair);
            return;
        }
    }
    dispatch_fused<S, 0>(h, pair);
}

}  // namespace eng
}  // namespace bgk
