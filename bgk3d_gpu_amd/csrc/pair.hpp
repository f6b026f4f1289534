// Two time steps in one pass over HBM (handle API).
//
// A step streams every population in and out once and does about 2 flop per
// byte, so the one-step kernels of collide.hpp run at the HBM rate and no
// faster.  collide_pair reads a lattice once, takes two steps and writes the
// other lattice once.
//
// A block owns a column of the grid: kTileX = 64 cells in x, TY rows in y,
// and a range of planes k0..k1, which it walks upwards.  In plane kk it
// takes the first step for the tile and one cell around it (TY + 2 waves,
// one row each, and one wave for the two columns beside the rows), hands the
// 16 populations that move in x or y to their neighbours through LDS, and
// takes the second step for the tile in plane kk - 1: the populations that
// move up (c_z = +1) were handed over two planes ago, those that stay in
// their plane one plane ago, those that move down just now.  What a cell has
// received waits in its thread's registers, so LDS holds one plane (two with
// double buffering, which saves the second barrier).
//
// The first step is taken twice for cells within one cell of a tile's border
// (with 13 rows, 64 x 13 tiles: 16 waves for 13 rows, and 2 planes more per
// block), their reads from L2: the tiles of one XCD are neighbours and walk up
// together, and HBM is read 1.09 times (FETCH_SIZE, 256^3 FP32).
//
// Measured at 256^3 FP32, us per step: 268 (410 with one step per launch), of
// which arithmetic and exchange alone take 78, without the loads 136, without
// the stores 161; the two streams run at 4.9 TB/s together.  Without the side
// columns (one value used per 128-byte line, 570 of 1274 line requests a
// plane) it takes 235.  Loads issued two planes ahead, or before the first
// step instead of after it, gave no more; plain stores 290, 6 waves and two
// blocks per CU 305, tiles in launch order over the XCDs 361.  FP64 at 192^3:
// 207 (359).
//
// Where at most 32 cells of a row are left, tiles of 32 cells with two rows
// per wave take them (half the waves of a 64-cell tile that is mostly empty):
// LES FP32 201 x 135 x 99 61 -> 56 us per step, FP32 87^3 18.4 -> 15.9, 130^3
// 50.0 -> 48.3, FP64 75^3 27.0 -> 22.8; 16 cells would no longer write whole
// FP32 lines.
//
// Each step is the one-step kernels' arithmetic on the same values, rounded
// to the storage type in between, so two steps here give the same bits as
// two there.  Boundaries are the same folded rules (collide.hpp); a bounced
// pull of the second step takes the thread's own opposite population of the
// first.  Direction 19 is read from one lattice and written to the other
// here (in place it would race with the border cells' reads).
#pragma once

#include <algorithm>
#include <cmath>

#include "collide.hpp"

namespace bgk {

constexpr int kTileX = 64;

// The tiles of a launch: tx * ty columns of 64 cells x th rows and, where the
// last 1 ... 32 cells of a row are left, ty2 columns of 32 cells x 2 th rows;
// each cut into cz ranges of zc planes.
struct PairGrid {
    int tx, ty, th, ty2, cz, zc;
    int total;  // (tx * ty + ty2) * cz
};

// Barrier of the block for LDS only: global loads stay in flight across it
// (__syncthreads would be free to wait for them).
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A wave-uniform address as a value of its own, in scalar registers: without
// it the compiler keeps a 64-bit address per lane and direction alive across
// the loop over the planes (22 registers more, and spills).
template <typename T>
__device__ __forceinline__ T* scalar_base(T* p)
{
    asm("" : "+s"(p));
    return p;
}

// A lane's 32-bit offset as a value formed here and now: its widening to 64
// bits then stays beside the load, where it folds into the instruction's
// scalar base + 32-bit offset form.
__device__ __forceinline__ uint32_t lane_offset(uint32_t v)
{
    asm("" : "+v"(v));
    return v;
}

// The exchange in LDS holds stored values as plain bits, through pointers in
// the LDS address space: with generic pointers the compiler turned "bounced ?
// own value : neighbour's" into one flat load from a selected pointer, the own
// value in scratch memory -- which faulted.
template <size_t N>
struct BitsOf;
template <>
struct BitsOf<4> {
    typedef uint32_t type;
};
template <>
struct BitsOf<8> {
    typedef uint64_t type;
};
#define BGK_LDS __attribute__((address_space(3)))

// Slot of direction d in the LDS exchange: the 16 directions that move in x
// or y; directions 6, 15 and 19 (d = 5, 14, 18) stay with their thread.
__host__ __device__ constexpr int lds_slot(int d) { return d < 5 ? d : (d < 14 ? d - 1 : d - 2); }
__device__ constexpr int kMid[9] = {0, 2, 4, 7, 9, 11, 13, 16, 18};  // directions with c_z = 0
template <int N>
__host__ __device__ constexpr int place(const int (&list)[N], int d)
{
    for (int q = 0; q < N; ++q)
        if (list[q] == d) return q;
    return -1;
}
__host__ __device__ constexpr bool stays(int d) { return cx_of(d) == 0 && cy_of(d) == 0; }

// One BGK step with the shifted storage's constants and the handle API's
// forces known at compile time: bgk_collide_ref without the terms that are
// zero there (cte0 = 0, the force components the mode does not set).  A term
// v + 0 differs from v only for v = -0: q = -0 gives e = s +- 0 with s = +0 or
// s != 0 either way, and a relaxed value x - omega (x - e) is -0 only for e =
// -0, which rp (...) + s never is.
// Each value goes to sink(std::integral_constant<int, d>{}, value) as soon as
// it is formed, opposite directions together, so that few are live at once
// (with LES every equilibrium is needed first).
template <typename R, int FMODE, bool LES, typename Sink>
__device__ __forceinline__ void bgk_collide_shifted(const R (&x)[19], R omega, R fgrad, R cte_s, Sink&& sink)
{
    const R p0 = W<R>::p0, p1 = W<R>::p1, p2 = W<R>::p2, three = R(3), qf = R(1.5);
    const R rho = density_ref(x, R(1));
    const R rhoinv = R(1) / rho;
    const R vx = (x[0] + x[1] + x[2] + x[3] + x[4] - x[9] - x[10] - x[11] - x[12] - x[13]) * rhoinv;
    const R vy = (x[2] + x[6] + x[7] + x[8] + x[11] - x[0] - x[9] - x[15] - x[16] - x[17]) * rhoinv;
    const R vz = (x[3] + x[5] + x[6] + x[12] + x[17] - x[1] - x[8] - x[10] - x[14] - x[15]) * rhoinv;
    const R vx2 = vx * vx, vy2 = vy * vy, vz2 = vz * vz;
    const R vsq = vx2 + vy2 + vz2;
    const R rp0 = rho * p0, rp1 = rho * p1, rp2 = rho * p2;
    const R s2 = rp2 - p2, s1 = rp1 - p1, s0 = rp0 - p0;
    const R force = fgrad * rho;
    auto emit = [&](auto dc, R e) {
        constexpr int d = decltype(dc)::value;
        constexpr int c = FMODE == 1 ? cx_of(d) : (FMODE == 2 ? cy_of(d) : (FMODE == 3 ? cz_of(d) : 0));
        const R v = x[d] - omega * (x[d] - e);
        sink(dc, c > 0 ? v + force : (c < 0 ? v - force : v));
    };
    // the equilibria of every pair of opposite directions, handed to f(d, e)
    auto equilibria = [&](auto&& f) {
        auto diagonal = [&](R v, auto dc) {
            const R r = three * v, q = qf * (r * v - vsq);
            f(dc, rp2 * (r + q) + s2);
            f(DirC<opp_of(decltype(dc)::value)>{}, rp2 * (-r + q) + s2);
        };
        auto axis = [&](R v, R v2, auto dc) {
            const R r = three * v, q = qf * (three * v2 - vsq);
            f(dc, rp1 * (r + q) + s1);
            f(DirC<opp_of(decltype(dc)::value)>{}, rp1 * (-r + q) + s1);
        };
        diagonal(vx - vy, DirC<0>{});
        diagonal(vx - vz, DirC<1>{});
        diagonal(vx + vy, DirC<2>{});
        diagonal(vx + vz, DirC<3>{});
        axis(vx, vx2, DirC<4>{});
        axis(vz, vz2, DirC<5>{});
        diagonal(vy + vz, DirC<6>{});
        axis(vy, vy2, DirC<7>{});
        diagonal(vy - vz, DirC<8>{});
        f(DirC<18>{}, rp0 * (qf * (-vsq)) + s0);
    };
    if constexpr (LES) {
        R e[19];
        equilibria([&](auto dc, R v) { e[decltype(dc)::value] = v; });
        omega = les_omega(x, e, omega, cte_s);
        for_each_dir([&](auto dc) { emit(dc, e[decltype(dc)::value]); });
    } else {
        equilibria(emit);
    }
}

// The step of one cell, rounded to the storage type, in the form the one-step
// kernels use for S; each value goes to sink(d, value).
template <typename S, int FMODE, typename Sink>
__device__ __forceinline__ void pair_collide(const FusedArgs<S>& p, const typename Storage<S>::compute (&x)[19],
                                             Sink&& sink)
{
    bgk_collide_shifted<typename Storage<S>::compute, (FMODE & 3), (FMODE & 4) != 0>(
        x, p.omega, p.fgrad, p.cte_s, [&](auto dc, auto v) { sink(dc, Rounder<S, 0>::cvt(v, 0u)); });
}

// v where mask is all ones, +0 where it is 0 (a select of 19 values would be
// compiled into a branch around their arithmetic).
template <typename S>
__device__ __forceinline__ S masked(S v, uint32_t mask)
{
    if constexpr (sizeof(S) == 8)
        return __builtin_bit_cast(S, __builtin_bit_cast(uint64_t, v) & ((uint64_t)mask << 32 | mask));
    else
        return __builtin_bit_cast(S, __builtin_bit_cast(uint32_t, v) & mask);
}

// Stored bits of a value, as the loads of this kernel return them.
template <typename S>
__device__ __forceinline__ S load_raw(const S* p)
{
    if constexpr (std::is_same<S, mix32_t>::value)
        return mix32_t{gmem(p)->v};
    else
        return *gmem(p);
}

// Tile rows a block can hold and its LDS buffers.  One block runs per CU
// (LDS, and 16 or 12 waves by their registers), so as many rows as fit:
// FP32 13 (16 waves of up to 128 registers, two 63 KB buffers); with FP64
// arithmetic 12 waves of up to 168 registers, 8 rows in FP64 storage (85 KB,
// so a single buffer) and 9 in FP32 (MIXED2).
template <typename S>
struct PairShape {
    static constexpr bool wide = std::is_same<typename Storage<S>::compute, double>::value;
    static constexpr int TY = sizeof(S) == 8 ? 8 : (wide ? 9 : 13);
    static constexpr bool DB = sizeof(S) < 8;
    static constexpr int POP = (TY + 2) * (kTileX + 2);  // LDS elements per population
};

// Storage types that take two steps per launch where that is faster (prefer_pair).
template <typename S>
constexpr bool kPairs = sizeof(S) >= 4;

// Two steps of the tile of 64 / RW cells x th rows whose first cell is (x0, j0,
// k0); with RW = 2 a wave holds two rows.  `lone`: the tile spans the row.
template <typename S, int BX, int BY, int BZ, bool OBST, int FMODE, bool NT, int RW>
__device__ __forceinline__ void pair_rows(const FusedArgs<S>& p, BGK_LDS typename BitsOf<sizeof(S)>::type* lds, int x0,
                                          int j0, int k0, int th, int zc, bool lone)
{
    constexpr int TY = PairShape<S>::TY;
    constexpr bool DB = PairShape<S>::DB;
    typedef typename Storage<S>::compute C;
    constexpr long ES = (long)sizeof(S);
    constexpr int TILE = kTileX / RW, ROWS = TY + 2, PITCH = TILE + 2, POP = PairShape<S>::POP, BUF = 16 * POP;
    static_assert((RW * TY + 2) * PITCH <= POP && 2 * (RW * TY + 2) <= 64, "LDS rows and side lanes");
    constexpr bool ZWALL = BZ == AX_WALL || BZ == AX_LID;
    constexpr bool BOUNCE = BX == AX_WALL || BY == AX_WALL || OBST;  // bounces that differ between lanes
    typedef typename BitsOf<sizeof(S)>::type Bits;

    const int k1 = k0 + zc - 1 < p.n ? k0 + zc - 1 : p.n;
    const int first = ZWALL && k0 == 1 ? 1 : k0 - 1, last = k1 + 1;
    const int end1 = ZWALL && last > p.n ? p.n : last;  // last plane of the first step

    // The thread's cell of the first step: LDS row r (0 and rows + 1 around
    // the tile), column c (0 and width + 1 around it).  Lanes past the row's
    // end, past the last row or past the side columns repeat another lane's
    // cell, so no lane is masked; cells outside a wall are computed on a cell
    // inside and unused.  With two rows per wave, wave 0 holds the rows below
    // and above the tile.
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int width = p.l - x0 + 1 < TILE ? p.l - x0 + 1 : TILE;
    const int rows = p.m - j0 + 1 < th ? p.m - j0 + 1 : th;
    const int col = lane & (TILE - 1);
    const bool side = wave == ROWS;
    const int jr = j0 - 1 + wave;  // RW = 1: the row of a wave that is not `side`
    int r = wave;
    bool out = !side && wave >= 1 && wave <= rows;
    bool helps = side ? !(BX == AX_WALL && lone)
                      : wave <= rows + 1 && (BY == AX_WALL ? jr >= 1 && jr <= p.m : jr <= p.m + 1);
    if constexpr (RW == 2) {
        r = wave == 0 ? (lane < TILE ? 0 : rows + 1) : 2 * wave - 1 + (lane < TILE ? 0 : 1);
        if (wave != 0 && r > rows) r -= 1;
        out = !side && wave >= 1 && 2 * wave - 1 <= rows;
        helps = side ? helps : wave == 0;
    }
    if (side) r = lane < 2 * (rows + 2) ? lane >> 1 : 0;
    const int c = side ? ((lane & 1) ? width + 1 : 0) : (col < width ? col + 1 : width);
    int i = x0 - 1 + c, j = j0 - 1 + r, face = 0;
    if (i < 1 || i > p.l) {
        if (BX == AX_HALO) face = i < 1 ? 1 : 2;
        i = (BX == AX_PERIODIC) == (i < 1) ? p.l : 1;
    }
    if (j < 1 || j > p.m) j = j < 1 ? p.m : (j == p.m + 1 ? 1 : p.m);
    const int jout = RW == 2 ? j : jr;  // the row of an `out` wave's lane, scalar with one row per wave
    const int at = r * PITCH + c;

    // Pulls of the first step: population d of plane k at base(d) + a 32-bit
    // offset per lane.  `cell` is the cell itself; `bias` keeps the offsets
    // of bounced pulls, which lie on another plane or population, positive.
    const long bias = (20 * p.pstride + p.nxy) * ES;
    const uint32_t cell = (uint32_t)(((long)j * p.nx + i) * ES + bias);
    const int xm = BX == AX_PERIODIC && i == 1 ? p.l - 1 : -1, xp = BX == AX_PERIODIC && i == p.l ? 1 - p.l : 1;
    const int ym = BY == AX_PERIODIC && j == 1 ? (p.m - 1) * p.nx : -p.nx;
    const int yp = BY == AX_PERIODIC && j == p.m ? (1 - p.m) * p.nx : p.nx;
    // Whether direction d bounces off an x or y wall at (iw, jw), the cell's
    // i and j, each plane as values of its own (lane_offset): the compiler
    // otherwise keeps a 64-lane mask per direction in scalar registers
    // across the planes, more than there are.
    auto wall = [&](int d, int iw, int jw) {
        return (BX == AX_WALL && ((cx_of(d) > 0 && iw == 1) || (cx_of(d) < 0 && iw == p.l))) ||
               (BY == AX_WALL && ((cy_of(d) > 0 && jw == 1) || (cy_of(d) < 0 && jw == p.m)));
    };
    // Obstacle links of the cell in plane k; only rows and planes of the box
    // look (the same for a whole wave).
    const bool boxed = OBST && x0 + TILE >= p.oi0 && x0 - 1 < p.oi0 + p.oni && j0 - 1 < p.oj0 + p.onj &&
                       j0 + th >= p.oj0;
    auto links = [&](int k) -> uint32_t {
        const unsigned ri = (unsigned)(i - p.oi0), rj = (unsigned)(j - p.oj0), rk = (unsigned)(k - p.ok0);
        if (ri < (unsigned)p.oni && rj < (unsigned)p.onj && rk < (unsigned)p.onk)
            return p.obits[(long)ri + (long)p.oni * ((long)rj + (long)p.onj * rk)];
        return 0;
    };
    auto in_box = [&](int k) { return OBST && boxed && (unsigned)(k - p.ok0) < (unsigned)p.onk; };
    auto load_plane = [&](int k, auto LINKS, uint32_t ob, S (&raw)[19]) {
        const int kb = BZ == AX_PERIODIC && k == 1 ? p.n : k - 1, kt = BZ == AX_PERIODIC && k == p.n ? 1 : k + 1;
        const char* below = scalar_base(reinterpret_cast<const char*>(p.a[0] + p.nxy * kb) - bias);
        const char* here = scalar_base(reinterpret_cast<const char*>(p.a[0] + p.nxy * k) - bias);
        const char* above = scalar_base(reinterpret_cast<const char*>(p.a[0] + p.nxy * kt) - bias);
        const char* resting = scalar_base(reinterpret_cast<const char*>(p.a[18] + p.nxy * k) - bias);
        const uint32_t own = lane_offset(cell);
        const int iw = (int)lane_offset((uint32_t)i), jw = (int)lane_offset((uint32_t)j);
        for_each_dir([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            constexpr int cx = cx_of(d), cy = cy_of(d), cz = cz_of(d);
            constexpr bool XY = (BX == AX_WALL && cx != 0) || (BY == AX_WALL && cy != 0) || decltype(LINKS)::value;
            const int ks = cz > 0 ? kb : (cz < 0 ? kt : k);
            const char* base = d == 18 ? resting : (cz > 0 ? below : (cz < 0 ? above : here)) + d * p.pstride * ES;
            uint32_t off = own + (uint32_t)(((cx > 0 ? xm : (cx < 0 ? xp : 0)) + (cy > 0 ? ym : (cy < 0 ? yp : 0))) *
                                            (int)ES);
            if constexpr (d < 18 && XY && cz != 0 && BZ == AX_PERIODIC) {
                // own opposite population: across the periodic seam too far for the 32-bit offset
                const char* from = base + (uint64_t)off;
                const char* mine = here + opp_of(d) * p.pstride * ES + (uint64_t)own;
                if (wall(d, iw, jw) || (decltype(LINKS)::value && ((ob >> d) & 1u))) from = mine;
                raw[d] = load_raw<S>(reinterpret_cast<const S*>(from));
                return;
            }
            if constexpr (d < 18 && (XY || (ZWALL && cz != 0))) {
                const bool zb = ZWALL && cz != 0 && (ks < 1 || ks > p.n);
                const long back = ((opp_of(d) - d) * p.pstride + cz * p.nxy) * ES;
                if (zb || wall(d, iw, jw) || (decltype(LINKS)::value && ((ob >> d) & 1u)))
                    off = own + (uint32_t)back;
            }
            raw[d] = load_raw<S>(reinterpret_cast<const S*>(base + (uint64_t)off));
        });
    };
    auto plane = [&](int kk) { return kk < 1 ? kk + p.n : (kk > p.n ? kk - p.n : kk); };

    S raw[19];           // plane kk as loaded, for the first step
    uint32_t ob = 0;     // link mask of the cell in that plane
    auto fetch = [&](int kk) {
        const int k = plane(kk);
        ob = 0;
        if constexpr (OBST) {
            if (in_box(k)) {
                ob = links(k);
                load_plane(k, std::true_type{}, ob, raw);
                return;
            }
        }
        load_plane(k, std::false_type{}, 0u, raw);
    };
    // First step of plane kk, and its part of the exchange.
    auto step_one = [&](int kk, BGK_LDS Bits* buf, S (&v)[19]) {
        C x[19];
        for_each_dir([&](auto dc) {
            constexpr int d = decltype(dc)::value;
            x[d] = Storage<S>::widen(raw[d]);
            if constexpr (BZ == AX_LID) x[d] = lid_value<S, d>(x[d], cz_of(d) < 0 && kk == p.n, p.lidforce);
        });
        pair_collide<S, FMODE>(p, x, [&](auto dc, S w) {
            constexpr int d = decltype(dc)::value;
            v[d] = w;
            if constexpr (!stays(d) && BX != AX_HALO) buf[lds_slot(d) * POP + at] = __builtin_bit_cast(Bits, w);
        });
        if constexpr (BX == AX_HALO) {
            if (face == 1) {
                S h[5];
                inflow_face<S>(p.uin, h);
                for (int d = 0; d < 5; ++d) v[d] = h[d];
            } else if (face == 2) {
                C f[19];
                for (int d = 0; d < 19; ++d) f[d] = Storage<S>::widen(v[d]);
                S h[5];
                outflow_face<S>(f, h);
                for (int d = 0; d < 5; ++d) v[9 + d] = h[d];
            }
            for_each_dir([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                if constexpr (!stays(d)) buf[lds_slot(d) * POP + at] = __builtin_bit_cast(Bits, v[d]);
            });
        }
    };
    auto buffer = [&](int kk) { return lds + (DB && (kk & 1) ? BUF : 0); };

    if (!out) {
        if (helps) {
            S v[19];
            fetch(first);
            for (int kk = first; kk <= end1; ++kk) {
                step_one(kk, buffer(kk), v);
                if (kk < end1) fetch(kk + 1);
                lds_barrier();
                if (!DB) lds_barrier();
            }
            if (end1 < last) lds_barrier();
        } else {
            for (int kk = first; kk <= last; ++kk) {
                lds_barrier();
                if (!DB && kk <= end1) lds_barrier();
            }
        }
        return;
    }

    // Rows of the second step.  Received and waiting: up (c_z > 0, for plane
    // kk), upn (c_z > 0, for kk - 1), mid (c_z = 0, for kk - 1); `ups`: the
    // cell's own c_z > 0 populations of plane kk - 1, for bounced pulls.
    S up[5], upn[5], mid[9], ups[5];
    uint32_t ob1 = 0;  // link mask in plane kk - 1
    constexpr int UP[5] = {3, 5, 6, 12, 17}, DN[5] = {10, 14, 15, 1, 8};
    const int lend = p.lend > p.l ? p.lend : p.l;
    const int ic = x0 + col < lend ? x0 + col : lend;
    const uint32_t live = ic <= p.l ? ~0u : 0u;
    const uint32_t to = (uint32_t)(((long)j * p.nx + ic) * ES);

    // One plane: STEP1 takes the first step of plane kk, STEP2 the second of
    // plane kk - 1.
    auto advance = [&](int kk, auto STEP1, auto STEP2) {
        constexpr bool S1 = decltype(STEP1)::value, S2 = decltype(STEP2)::value;
        BGK_LDS Bits* buf = buffer(kk);
        S v[19];
        const uint32_t ob0 = ob;
        const int iw = (int)lane_offset((uint32_t)i), jo = RW == 2 ? (int)lane_offset((uint32_t)jout) : jout;
        if constexpr (S1) {
            step_one(kk, buf, v);
            if constexpr (BOUNCE || ZWALL) {  // bounced pulls of plane kk from below: own populations going down
                for (int q = 0; q < 5; ++q) {
                    const int d = UP[q];
                    if ((ZWALL && kk == 1) || wall(d, iw, jo) || (OBST && ((ob0 >> d) & 1u))) up[q] = v[DN[q]];
                }
            }
            if (kk < end1) fetch(kk + 1);
        }
        lds_barrier();
        auto get = [&](auto dc) -> S {
            constexpr int d = decltype(dc)::value;
            return __builtin_bit_cast(S, (Bits)buf[lds_slot(d) * POP + at - cy_of(d) * PITCH - cx_of(d)]);
        };
        if constexpr (S2) {
            C x[19];
            for_each_dir([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                S w;
                if constexpr (cz_of(d) > 0) {
                    w = upn[place(UP, d)];
                } else if constexpr (cz_of(d) == 0) {
                    w = mid[place(kMid, d)];
                } else {
                    constexpr int q = place(DN, d);
                    if constexpr (!S1) {
                        w = ups[q];
                    } else {
                        if constexpr (stays(d))
                            w = v[d];
                        else
                            w = get(dc);
                        if constexpr (BOUNCE)
                            if (wall(d, iw, jo) || (OBST && ((ob1 >> d) & 1u))) w = ups[q];
                    }
                }
                x[d] = Storage<S>::widen(w);
                if constexpr (BZ == AX_LID && !S1) x[d] = lid_value<S, d>(x[d], cz_of(d) < 0, p.lidforce);
            });
            // whole lines: the lanes past the row up to lend store zeros (the lanes past that repeat the last)
            char* moving = scalar_base(reinterpret_cast<char*>(p.b[0] + p.nxy * (kk - 1)));
            char* resting = scalar_base(reinterpret_cast<char*>(p.brest + p.nxy * (kk - 1)));
            const uint32_t off = lane_offset(to);
            pair_collide<S, FMODE>(p, x, [&](auto dc, S w) {
                constexpr int d = decltype(dc)::value;
                char* base = d == 18 ? resting : moving + d * p.pstride * ES;
                store_to<NT>(reinterpret_cast<S*>(base + (uint64_t)off), masked(w, live));
                if constexpr (d == 18) flag_nonfinite(p, Storage<S>::widen(w));
            });
        }
        if constexpr (S1) {
            for_each_dir([&](auto dc) {
                constexpr int d = decltype(dc)::value;
                if constexpr (cz_of(d) == 0) {
                    S w = v[18];
                    if constexpr (d != 18) {
                        // bounced: the own opposite value, from LDS too (kept in registers
                        // across the barrier it cost spills: FP64 cavity 256^3 543 -> 469 us)
                        int q = lds_slot(d) * POP + at - cy_of(d) * PITCH - cx_of(d);
                        if constexpr (BOUNCE)
                            if (wall(d, iw, jo) || (OBST && ((ob0 >> d) & 1u))) q = lds_slot(opp_of(d)) * POP + at;
                        w = __builtin_bit_cast(S, (Bits)buf[q]);
                    }
                    mid[place(kMid, d)] = w;
                } else if constexpr (cz_of(d) > 0) {
                    constexpr int q = place(UP, d);
                    upn[q] = up[q];
                    if constexpr (stays(d))
                        up[q] = v[d];
                    else
                        up[q] = get(dc);
                    if constexpr (BOUNCE || ZWALL) ups[q] = v[d];
                }
            });
        }
        ob1 = ob0;
        if (!DB && S1) lds_barrier();
    };
    typedef std::true_type T;
    typedef std::false_type F;
    fetch(first);
    for (int kk = first; kk <= k0; ++kk) advance(kk, T{}, F{});
    // The loop's first pass is written out: on entry to the loop the loads of
    // the next plane are then followed by 19 stores on either path, and the
    // compiler's waits for those loads leave the stores in flight.
    if (k0 < end1) {
        advance(k0 + 1, T{}, T{});
        for (int kk = k0 + 2; kk <= end1; ++kk) advance(kk, T{}, T{});
    }
    if (end1 < last) advance(last, F{}, T{});
}

// Two steps of one tile of the launch.
template <typename S, int BX, int BY, int BZ, bool OBST, int FMODE, bool NT = true>
__device__ __forceinline__ void pair_tile(const FusedArgs<S>& p, const PairGrid& g, int tile)
{
    typedef typename BitsOf<sizeof(S)>::type Bits;
    __shared__ Bits lds_[(PairShape<S>::DB ? 2 : 1) * 16 * PairShape<S>::POP];
    BGK_LDS Bits* const lds = (BGK_LDS Bits*)lds_;
    const int per = g.tx * g.ty + g.ty2, q = tile % per;
    const int k0 = 1 + (tile / per) * g.zc;
    const bool lone = g.tx + (g.ty2 ? 1 : 0) == 1;
    if (q < g.tx * g.ty)
        pair_rows<S, BX, BY, BZ, OBST, FMODE, NT, 1>(p, lds, 1 + q % g.tx * kTileX, 1 + q / g.tx * g.th, k0, g.th, g.zc,
                                                 lone);
    else
        pair_rows<S, BX, BY, BZ, OBST, FMODE, NT, 2>(p, lds, 1 + g.tx * kTileX, 1 + (q - g.tx * g.ty) * 2 * g.th, k0,
                                                 2 * g.th, g.zc, lone);
}

// Block x of n blocks as the b-th tile: consecutive tiles on one XCD (blocks
// go to the 8 XCDs in turn).  May return n or more: no tile.
__device__ __forceinline__ int xcd_tile(int x, int n)
{
    const int per = (n + 7) / 8;
    return (x >> 3) < per ? (x & 7) * per + (x >> 3) : n;
}

template <typename S, int BX, int BY, int BZ, bool OBST, int FMODE, bool NT = true>
__global__ __launch_bounds__(64 * (PairShape<S>::TY + 3)) void collide_pair(FusedArgs<S> p, PairGrid g)
{
    const int tile = xcd_tile((int)blockIdx.x, g.total);
    if (tile < g.total) pair_tile<S, BX, BY, BZ, OBST, FMODE, NT>(p, g, tile);
}

// Tiles of an l x m x n lattice with at most `rows` rows: the rows and planes
// per block that minimise `cost`, the time of a launch in units of one row of
// 64 cells taken one plane on.  A block takes zc + 2 planes of th + 2 rows
// (a fit has smaller constants, since the border rows and first planes do
// less); `cus` blocks run at a time (256, one per CU, in a launch of its own).
// One round of blocks is worth a lot: tiles that walk up together share their
// border reads in L2 and no CU waits for a block to start, so two full rounds
// cost 2.3 of one, and a launch of 257 blocks 1.7 (900 x 150^2 FP32, per
// step: 247 blocks 323 us, the same columns cut in two 365, in five 376;
// 400^3: 241 blocks 1030 us, 404 1359, 1010 1230).  The weights fit 45 such
// launches (256^3, 400^3, 512^3, 900 x 150^2) to 8 %.
inline PairGrid pair_grid(int l, int m, int n, int rows, double& cost, double cus = 256)
{
    PairGrid g{};
    const int left = l % kTileX;
    const bool tail = left > 0 && left <= kTileX / 2;
    g.tx = l / kTileX + (left > kTileX / 2 ? 1 : 0);
    cost = -1;
    for (int th = std::min(m, rows); th >= 1; --th) {
        const int ty = ceil_div(m, th);
        if (ceil_div(m, ty) != th) continue;  // as many tiles of fewer rows
        for (int zc = n, cz = 1;; cz = ceil_div(n, zc - 1), zc = ceil_div(n, cz)) {  // every distinct cut of n
            const int ty2 = tail ? ceil_div(m, 2 * th) : 0;
            const double blocks = ((double)g.tx * ty + ty2) * cz;
            if (blocks >= 1u << 30) break;
            const double rounds = blocks / cus;
            const double c = (rounds <= 1 ? 0.9 + 0.1 * rounds : 0.55 * std::ceil(rounds) + 0.62 * rounds) * (zc + 1) *
                             (th + 2.5);
            if (cost < 0 || c < cost) {
                cost = c;
                g.ty = ty;
                g.th = th;
                g.ty2 = ty2;
                g.cz = cz;
                g.zc = zc;
                g.total = (int)blocks;
            }
            if (zc == 1) break;
        }
    }
    return g;
}

// Tiles of `rows` rows (at most the kernel's TY) and `planes` planes.
inline PairGrid pair_grid_of(int l, int m, int n, int rows, int planes)
{
    PairGrid g{};
    const int left = l % kTileX;
    const bool tail = left > 0 && left <= kTileX / 2;
    g.tx = l / kTileX + (left > kTileX / 2 ? 1 : 0);
    g.th = rows;
    g.ty = ceil_div(m, rows);
    g.ty2 = tail ? ceil_div(m, 2 * rows) : 0;
    g.zc = planes;
    g.cz = ceil_div(n, planes);
    const double blocks = ((double)g.tx * g.ty + g.ty2) * g.cz;
    g.total = blocks < 1u << 30 ? (int)blocks : 0;
    return g;
}

inline int pair_blocks(int tiles) { return ceil_div(tiles, 8) * 8; }

template <typename S, int BX, int BY, int BZ, bool OB, int FM, bool NT = true>
void launch_pair(const FusedArgs<S>& p, const PairGrid& g, hipStream_t stream)
{
    hipLaunchKernelGGL((collide_pair<S, BX, BY, BZ, OB, FM, NT>), dim3((unsigned)pair_blocks(g.total)),
                       dim3(64 * (PairShape<S>::TY + 3)), 0, stream, p, g);
}

}  // namespace bgk
