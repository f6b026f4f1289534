// Internals shared by the handle API (engine.hip) and the serving layer
// (serving.hip): the handle, its layout, the derived collision parameters
// and the arguments of the fused kernel for one step.
#pragma once

#include "../../include/bgk3d_engine.h"

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "collide.hpp"
#include "common.hpp"
#include "d3q19.hpp"
#include "pair.hpp"
#include "reduce.hpp"
#include "storage.hpp"
#include "v1_kernels.hpp"

struct bgk_handle {
    bgk_config cfg{};
    size_t esize = 4;
    int A = 32;  // elements per 128-byte line
    // Layout of a lattice: the population planes of one z level lie next to
    // each other, population d of cell (i,j,k) at
    //   mem[buf] + base + d*plane + i + nx*j + nxy*k,
    // plane = nx*ny, z stride nxy = 19*plane.  Direction 19 is in lattice
    // `rest`: single steps update it in place, pairs of steps move it to the
    // other lattice's slot.  Rows are padded to whole 128-byte
    // lines and base puts i = 1 on a line start.  A wave's 19 loads and 19
    // stores then fall in two windows of 19 planes instead of 37 arrays
    // scattered over the whole region: fewer DRAM pages and translation
    // entries in flight per step.
    int nx = 0, ny = 0, nz = 0;
    long plane = 0, nxy = 0, lstride = 0, base = 0;
    // compact layout: rows of l + 2 cells (collide_compact), else rows padded
    // to whole lines (collide_fused)
    bool compact = false;
    // two steps per launch (collide_pair) where two are left, in tiles pgrid.
    // `flex`: one step at a time would run on compact rows; lstride holds a
    // lattice of either rows (relayout)
    bool pair = false, flex = false;
    int launch = 0;   // steps per launch asked for (bgk_set_launch), 0: the rule's
    double owed = 0;  // steps that the other rows would have saved (choose_rows)
    bgk::PairGrid pgrid{};
    void* mem[2] = {nullptr, nullptr};
    size_t bytes = 0;
    int cur = 0, rest = 0;
    hipStream_t stream = nullptr;
    double omega = 0, fgrad = 0, lidforce = 0, u_inflow = 0, cte_s = 0;
    // obstacle
    bool has_obs = false;
    int ic = 0, jc = 0, kc = 0, radius = 0;
    int ob[6] = {0, 0, 0, 0, 0, 0};  // link-mask box origin (i,j,k) and extent
    uint32_t* obits = nullptr;
    int mk[6] = {0, 0, 0, 0, 0, 0};  // solid-mask box origin and extent (draglift)
    int8_t* omask = nullptr;
    double* scratch = nullptr;
    double* hscratch = nullptr;
    // device and pinned host staging of bgk_fields, from its first call on;
    // one call at a time uses (and may replace) it
    std::mutex stage_lock;
    void *stage = nullptr, *hstage = nullptr;
    size_t stage_bytes = 0;
    long long steps = 0;
    bool borrowed = false;  // lattice memory, scratch and stream belong to a server
    std::vector<hipEvent_t> events;

    template <typename S>
    S* arr(int buf, int d) const
    {
        return reinterpret_cast<S*>(mem[buf]) + (long)d * plane + base;
    }
    template <typename S>
    S* cur_a(int d) const
    {
        return arr<S>(d == 18 ? rest : cur, d);
    }
    template <typename S>
    bgk::Lattice19<S> current() const
    {
        bgk::Lattice19<S> L;
        for (int d = 0; d < 19; ++d) L.p[d] = cur_a<S>(d);
        return L;
    }
    bgk::Geometry geom() const
    {
        bgk::Geometry g;
        g.l = cfg.l;
        g.m = cfg.m;
        g.n = cfg.n;
        g.nx = nx;
        g.nxy = nxy;
        return g;
    }
};

namespace bgk {
namespace eng {

// Record an error message for bgk_last_error() and return `code`.
int fail(int code, const char* fmt, ...);

#define ENG_HIP(call)                                                                                    \
    do {                                                                                                 \
        hipError_t _e = (call);                                                                          \
        if (_e != hipSuccess) return ::bgk::eng::fail(BGK_EHIP, "%s: %s", #call, hipGetErrorString(_e)); \
    } while (0)

// Drop the HIP error that an earlier call of this thread left (a handle that
// did not fit, another library's query): the launch checks read the last one.
inline void forget_error() { (void)hipGetLastError(); }

inline size_t storage_bytes(int kind)
{
    switch (kind) {
        case BGK_F32: return 4;
        case BGK_F64: return 8;
        default: return 2;
    }
}

inline long round_up(long v, long a) { return (v + a - 1) / a * a; }

// Row layout of the automatic choice (layout = 0).  Measured kernel times,
// compact/padded (cavities, Taylor-Green and channels alone, one handle):
//  * FP32 and FP64: 0.94-0.99 from 3.5 % row waste up (n = 100 ... 250),
//    even at 2 %; at zero waste 1.09-1.14 at 64^3, 1.00-1.04 from 96^3 to
//    224^3, 0.94-0.99 from 256^3 up (384^3, 1024 x 384^2, 512 x 512 x 256).
//  * 16-bit storage: 0.86-0.99 from 10 % waste up, even at 6-8 %, 1.04-1.07
//    at 2-4 % (n = 184, 188, 250) and 1.06-1.13 at zero waste (256^3), 0.97
//    at 384^3.
inline bool prefer_compact(const bgk_config& c, double waste)
{
    const bool wide = storage_bytes(c.storage) >= 4;
    if (waste > (wide ? 0.03 : 0.09)) return true;
    return wide && (double)c.l * (double)c.m * (double)c.n >= (double)(1 << 24);
}

// Calls f with a value of the storage type the configuration selects: the
// storage kind, or for the mixed forms the type that carries their
// collision kind (mix32_t, f16r_t).
template <typename F>
int by_storage(const bgk_config& c, F&& f)
{
    if (c.mixed == 2 && c.storage == BGK_F32) return f(mix32_t{});
    if (c.mixed == 1 && c.storage == BGK_F16) return f(f16r_t{});
    switch (c.storage) {
        case BGK_F32: return f(float{});
        case BGK_F64: return f(double{});
        case BGK_F16: return f(f16_t{});
        case BGK_BF16: return f(bf16_t{});
    }
    return fail(BGK_EINVAL, "unknown storage type %d", c.storage);
}

// The collision runs in FP64 (DOUBLE_P storage, or the MIXED2 form).
inline bool compute_double(const bgk_config& c) { return c.storage == BGK_F64 || c.mixed == 2; }

// Whether two steps per launch can be taken at all, on padded rows with
// `plane` values a population plane.
inline bool can_pair(const bgk_config& c, long plane)
{
    const size_t es = storage_bytes(c.storage);
    if (es < 4 || c.layout == 2) return false;
    // a lane's 32-bit byte offset spans up to four z levels (pair_tile)
    return 80.0 * (double)es * (double)plane < 4.0e9;
}

// Most rows of a tile.
inline int pair_rows_max(const bgk_config& c)
{
    return c.storage == BGK_F64 ? PairShape<double>::TY
                                : (compute_double(c) ? PairShape<mix32_t>::TY : PairShape<float>::TY);
}

// Tiles of the two-step kernel for this configuration, if two steps per
// launch are estimated to be faster than two launches of one.  Estimates in
// us: a single step takes 1.5 + its bytes at 6.2 TB/s, at least 4.6; a pair 2.5 +
// its cost (pair_grid) times 0.42 in FP32, 0.46 in MIXED2 and 0.70 in FP64; with
// LES 0.44, 0.53 and 1.10 (more values live than registers).  Both are fitted
// to lattices that stream: above 256 MB the pair's factors measured 0.38 ...
// 0.42, 0.39 ... 0.45, 0.55 ... 0.74 (LES 0.40 ... 0.47, 0.46 ... 0.54, 0.92 ... 1.15),
// a single step 1.00 ... 1.25 of its estimate.  From 80 to 256 MB, where the
// pair's stores stay in the cache (keep_in_cache), they are 0.28 ... 0.40, 0.34
// ... 0.44, 0.51 ... 0.63 (0.33 ... 0.44, 0.43 ... 0.54, 0.72 ... 0.95) and 1.05 ... 1.35, and
// below that they scatter: there the rule refuses lattices that two steps per
// launch would serve better.  Over 504 lattices (24^3 ... 200^3 and flat or long
// boxes, six forms, with bgk_set_launch) it took two only where that is faster,
// and refused it 201 times where it is by more than 3 %.  Measured per step, one
// step a launch against two: taken FP32 256^3 410 / 268, 150^3 88 / 64, 64^3 9.6 /
// 6.1, FP64 192^3 359 / 207, 80^3 29.4 / 18.3; LES 128^3 MIXED2 60.7 / 47.5, FP64
// 109 / 95; refused FP32 40^3 5.8 / 4.5, 80^3 17.6 / 11.8, 97^3 28.1 / 17.5, 100^3 29.6
// / 20.2, FP64 56^3 12.9 / 8.6, MIXED2 100^3 28.8 / 25.9, 140^3 LES MIXED2 77 / 71.
// 16-bit storage stays with one: its kernels are bound by issue as much as by
// HBM (FP16 channel at 512 x 128^2 108 / 118 with one cell per lane, 109 / 131
// with two).
inline bool prefer_pair(const bgk_config& c, long plane, PairGrid& g)
{
    if (!can_pair(c, plane)) return false;
    const size_t es = storage_bytes(c.storage);
    const bool wide = compute_double(c);
    double cost;
    g = pair_grid(c.l, c.m, c.n, pair_rows_max(c), cost);
    const double cells = (double)c.l * c.m * c.n;
    const double two = 2 * std::max(4.6, 1.5 + 38.0 * (double)es * cells / 6.2e6);
    const double us = es == 8 ? (c.les ? 1.10 : 0.70) : (wide ? (c.les ? 0.53 : 0.46) : (c.les ? 0.44 : 0.42));
    return 2.5 + cost * us < two;
}

// Validate `c` and fill the layout and the derived parameters of `h`
// (no device call, no allocation).  `roomy`: two steps per launch also where
// one step would run on compact rows, which need less memory than the padded
// rows of collide_pair (130^3 FP32: 21 %).
int handle_setup(bgk_handle& h, const bgk_config& c, bool roomy = true);

// Rows of the handle from here on: compact, or padded to whole lines.
inline void set_rows(bgk_handle& h, bool compact)
{
    h.compact = compact;
    if (compact) {
        // cell (0, 1, k) of every population plane on a line start
        h.nx = h.cfg.l + 2;
        h.plane = round_up((long)h.nx * h.ny, h.A);
        h.base = (h.A - h.nx % h.A) % h.A;
    } else {
        // cell (1, j, k) on a line start
        h.nx = (int)round_up(h.cfg.l + 2, h.A);
        h.plane = (long)h.nx * h.ny;
        h.base = h.A - 1;
    }
    h.nxy = 19 * h.plane;
}

// Queue the move of a flex handle's populations to the other rows, and of
// direction 19 to the lattice of the others (relayout does that too).
int relayout(bgk_handle& h, bool compact);
int join_rest(bgk_handle& h);

// Device bytes of the two lattices of a handle set up by handle_setup.
inline size_t lattice_bytes(const bgk_handle& h) { return (size_t)h.lstride * 2 * h.esize; }

// Whether the lattices a launch works on, `bytes` together, are stored with
// plain instead of streaming stores: the next step then finds them in the
// 256 MB last-level cache.  Above that streaming is faster, and below 80 MB
// too (two steps per launch, where prefer_pair refuses them by bgk_set_launch;
// us per step, streaming against plain: FP32 48^3 5.7 / 6.2, 64^3 6.4 / 6.7, 80^3
// 15.0 / 12.0, 100^3 25.0 / 20.2, 112^3 30.4 / 23.4, 128^3 (411 MB) 36.0 / 37.9; FP64
// 64^3 (106 MB) 10.7 / 10.8, 75^3 20.3 / 17.0, 90^3 30.7 / 25.0, 100^3 (354 MB) 43.0 /
// 45.7).
inline bool keep_in_cache(size_t bytes) { return bytes >= 80000000 && bytes <= size_t(1) << 28; }

// Point mem[0] and mem[1] (the two lattices) into one region of
// lattice_bytes(h) bytes.
inline void place_lattices(bgk_handle& h, void* region)
{
    h.mem[0] = region;
    h.mem[1] = static_cast<char*>(region) + (size_t)h.lstride * h.esize;
    h.bytes = lattice_bytes(h);
}

// Stochastic-rounding seed of the step that follows `steps` completed steps.
__host__ __device__ inline uint32_t step_seed(uint32_t cfg_seed, long long steps)
{
    return hash32(cfg_seed ^ hash32((uint32_t)steps * 0x9e3779b9U + 1u));
}

// Arguments of the fused kernel for the step that reads lattice `cur` and
// finds direction 19 in lattice `rest`.
template <typename S>
FusedArgs<S> fused_args(const bgk_handle& h, int cur, int rest)
{
    typedef typename Storage<S>::compute C;
    FusedArgs<S> p{};
    for (int d = 0; d < 19; ++d) p.a[d] = h.arr<S>(d == 18 ? rest : cur, d);
    p.brest = h.arr<S>(1 - rest, 18);
    for (int d = 0; d < 18; ++d) p.b[d] = h.arr<S>(1 - cur, d);
    p.l = h.cfg.l;
    p.m = h.cfg.m;
    p.n = h.cfg.n;
    p.nx = h.nx;
    p.nxy = h.nxy;
    p.omega = (C)h.omega;
    p.fgrad = (C)h.fgrad;
    p.fx = p.fy = p.fz = C(0);
    p.lidforce = (C)h.lidforce;
    p.cte_s = (C)h.cte_s;
    p.cst = CollideConsts<C>::shifted();
    p.obits = h.obits;
    p.oi0 = h.ob[0];
    p.oj0 = h.ob[1];
    p.ok0 = h.ob[2];
    p.oni = h.ob[3];
    p.onj = h.ob[4];
    p.onk = h.ob[5];
    p.align = 0;
    // padded rows start on a 128-byte line; with the x boundary folded into
    // the pull the cells after i = l up to that line's end are never read.
    // Compact rows: the positions the waves of a plane cover.
    if (h.compact)
        p.lend = (int)round_up((long)h.nx * h.cfg.m, h.A);
    else
        p.lend = h.cfg.boundary == BGK_BC_INFLOW ? 0 : (int)round_up(h.cfg.l, h.A);
    p.seed = step_seed(h.cfg.seed, h.steps);
    p.pstride = h.plane;
    p.uin = (C)h.u_inflow;
    return p;
}

// Queue the collide of the next step, or of the next two in one launch
// (launch.hpp).
template <typename S>
void launch_step(bgk_handle& h, bool pair);

}  // namespace eng
}  // namespace bgk
