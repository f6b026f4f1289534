// Handle API (include/bgk3d_engine.h): library-owned lattices laid out for
// gfx950, boundaries folded into the fused pull, FP32/FP64/FP16/BF16
// storage.
//
// Layout of one lattice: the reference's (0:nx-1, 0:ny-1, 0:nz-1) halo
// array per population, with nx rounded up to a multiple of A = 128 bytes /
// sizeof(storage) and the start shifted by A-1 elements, so the first
// interior cell of every row (i = 1) begins a 128-byte line: a wave's loads
// of the unshifted directions and all its stores then touch whole lines.
// The populations' z planes are interleaved (plane k of population d at
// (19 k + d) planes from the start), so one step's reads and writes move
// through two compact windows of the lattices instead of 37 separate
// arrays.  Directions 1..18 alternate between the two lattices (the
// reference's pointer swap, SRC/col_MC.F90:539-596), tracked by `cur`; so
// does direction 19 in a launch of two steps (collide_pair), tracked by
// `rest`, while a single step updates it in place.
#include "engine_internal.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "host_init.hpp"
#include "init_kernels.hpp"
#include "io_kernels.hpp"

using namespace bgk;
using namespace bgk::eng;

namespace bgk {
namespace eng {

namespace {
thread_local std::string g_err;
}

int fail(int code, const char* fmt, ...)
{
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return code;
}

const char* last_error() { return g_err.c_str(); }

}  // namespace eng
}  // namespace bgk


namespace {

// ---------------------------------------------------------------------------
// kernels specific to the engine
// ---------------------------------------------------------------------------

// Inflow halo x = 0, directions 1..5, every (j,k) incl. halo rows, the
// values of inflow_face.  Constant in time: with rows padded to whole lines
// the collide never writes a halo cell, and this runs once per lattice.
template <typename S>
__global__ void inflow_halo(Lattice19<S> a, Geometry g, typename Storage<S>::compute u_inflow)
{
    const int nj = g.m + 2;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nj * (g.n + 2)) return;
    const int j = t % nj, k = t / nj;
    S v[5];
    inflow_face<S>(u_inflow, v);
    const long s = gidx(g, 0, j, k);
    for (int d = 0; d < 5; ++d) store_value(a.p[d] + s, v[d]);
}

// Outflow halo x = l+1, directions 10..14, interior (j,k): outflow_face of
// cell (l,j,k).  The fused pull wraps j and k before reading this halo,
// which reproduces the reference's y/z periodic copies of the halo rows.
// Compact rows: the previous collide stored zeros over both x halos of this
// lattice unless it wrote the faces itself (kFillsInflowFaces), so `refill`
// also writes the inflow face x = 0 of the rows the pull reads (interior j,
// k), with the values inflow_halo writes.
template <typename S>
__global__ void outflow_halo(Lattice19<S> a, Geometry g, bool refill, typename Storage<S>::compute u_inflow)
{
    typedef typename Storage<S>::compute R;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= g.m * g.n) return;
    const int j = 1 + t % g.m, k = 1 + t / g.m;
    const long si = gidx(g, g.l, j, k);
    R f[19];
#pragma unroll
    for (int d = 0; d < 18; ++d) f[d] = Storage<S>::load(a.p[d] + si);
    f[18] = R(0);  // not used
    S v[5];
    outflow_face<S>(f, v);
    const long so = gidx(g, g.l + 1, j, k);
    for (int d = 0; d < 5; ++d) store_value(a.p[9 + d] + so, v[d]);
    if (refill) {
        inflow_face<S>(u_inflow, v);
        const long s0 = gidx(g, 0, j, k);
        for (int d = 0; d < 5; ++d) store_value(a.p[d] + s0, v[d]);
    }
}

// Direction 19 of one lattice into the other's place for it: `planes` z
// levels, `plane` values each, nxy apart.
template <typename S>
__global__ void move_rest(const S* __restrict__ from, S* __restrict__ to, long plane, long nxy, int planes)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= plane * planes) return;
    const long e = t % plane + t / plane * nxy;
    to[e] = from[e];
}

// A whole lattice into other rows: interior cells from `from`, zeros in the
// halo and in the row padding, which no folded boundary reads (planes of
// `plane` values, the halo ones among them).
template <typename S>
__global__ void move_rows(Lattice19<S> from, Geometry gf, Lattice19<S> to, Geometry gt, long plane)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= plane * (gt.n + 2)) return;
    const int k = (int)(t / plane), e = (int)(t % plane), j = e / gt.nx, i = e - j * gt.nx;
    const bool inside = i >= 1 && i <= gt.l && j >= 1 && j <= gt.m && k >= 1 && k <= gt.n;
    const long at = e + gt.nxy * k, src = inside ? gidx(gf, i, j, k) : 0;
#pragma unroll
    for (int d = 0; d < 19; ++d) to.p[d][at] = inside ? from.p[d][src] : S{};
}

// Momentum exchange over fluid cells of [is..ie]x[js..je]x[ks..ke]
// (SRC/draglift.F90:77-176); the solid mask is held for a box around the
// obstacle only (cells outside it are fluid).
template <typename S>
__global__ __launch_bounds__(kRedThreads) void draglift_box(Lattice19<S> a, Geometry g, const int8_t* __restrict__ om,
                                                            int mi0, int mj0, int mk0, int mni, int mnj, int mnk,
                                                            int is, int ie, int js, int je, int ks, int ke,
                                                            double* __restrict__ part)
{
    typedef typename Storage<S>::compute R;
    auto O = [&](int i, int j, int k) -> int {
        const unsigned ri = (unsigned)(i - mi0), rj = (unsigned)(j - mj0), rk = (unsigned)(k - mk0);
        if (ri >= (unsigned)mni || rj >= (unsigned)mnj || rk >= (unsigned)mnk) return 0;
        return om[(long)ri + (long)mni * ((long)rj + (long)mnj * rk)];
    };
    double v[3] = {0, 0, 0};
    const int ni = ie - is + 1, nj = je - js + 1, nk = ke - ks + 1;
    const long cells = (long)ni * nj * nk;
    for (long c = (long)blockIdx.x * kRedThreads + threadIdx.x; c < cells; c += (long)gridDim.x * kRedThreads) {
        const int i = is + (int)(c % ni), j = js + (int)((c / ni) % nj), k = ks + (int)(c / ((long)ni * nj));
        if (O(i, j, k) != 0) continue;
        const long s = gidx(g, i, j, k);
        R fxs = R(0), fys = R(0), fzs = R(0);
#pragma unroll
        for (int d = 0; d < 18; ++d) {
            const R ad = Storage<S>::load(a.p[d] + s);
            const R ob = (R)O(i + cx_of(d), j + cy_of(d), k + cz_of(d));
            const R tx = R(2.0) * (R)cx_of(d) * ad * ob;
            const R ty = R(2.0) * (R)cy_of(d) * ad * ob;
            const R tz = R(2.0) * (R)cz_of(d) * ad * ob;
            fxs = d == 0 ? tx : fxs + tx;
            fys = d == 0 ? ty : fys + ty;
            fzs = d == 0 ? tz : fzs + tz;
        }
        v[0] += (double)fxs;
        v[1] += (double)fys;
        v[2] += (double)fzs;
    }
    block_sum<3>(v);
    if (threadIdx.x == 0) {
        part[(long)blockIdx.x * 3 + 0] = v[0];
        part[(long)blockIdx.x * 3 + 1] = v[1];
        part[(long)blockIdx.x * 3 + 2] = v[2];
    }
}

// ---------------------------------------------------------------------------
// host helpers
// ---------------------------------------------------------------------------

bool sphere_solid(const bgk_handle& h, int i, int j, int k)
{
    if (!h.has_obs) return false;
    if (i < 1 || i > h.cfg.l || j < 1 || j > h.cfg.m || k < 1 || k > h.cfg.n) return false;
    const long d2 = (long)(h.ic - i) * (h.ic - i) + (long)(h.jc - j) * (h.jc - j) + (long)(h.kc - k) * (h.kc - k);
    const long R = h.radius;
    if (h.cfg.obstacle == 1) return d2 > (R - 2) * (R - 2) && d2 < (R + 2) * (R + 2);  // SRC/build.obs.F90:70-81
    return d2 <= R * R;                                                                // solid sphere
}

int wrap(int v, int n) { return v < 1 ? v + n : (v > n ? v - n : v); }

// The inflow face x = 0 of both lattices.
template <typename S>
void fill_inflow(bgk_handle& h)
{
    for (int buf = 0; buf < 2; ++buf) {
        Lattice19<S> L;
        for (int d = 0; d < 19; ++d) L.p[d] = h.arr<S>(buf, d);
        hipLaunchKernelGGL(inflow_halo<S>, dim3(ceil_div((long)(h.cfg.m + 2) * (h.cfg.n + 2), 256)), dim3(256), 0,
                           h.stream, L, h.geom(), (typename Storage<S>::compute)h.u_inflow);
    }
}

template <typename S>
int upload_state(bgk_handle& h)
{
    typedef typename Storage<S>::compute C;
    const bgk_config& c = h.cfg;
    // rest state: shifted populations are all zero, which the memset left
    if (c.init == 1 || c.init == 2) {
        // Taylor-Green: sin/cos factors per coordinate on the host, f_eq per
        // cell on the device (bit-identical to the host form), both lattices
        const C u00 = (C)(c.boundary == BGK_BC_CHANNEL ? 0.0 : c.u0);
        for (int buf = 0; buf < 2; ++buf) {
            S* ptrs[19];
            for (int d = 0; d < 19; ++d) ptrs[d] = (buf == 1 && d == 18) ? nullptr : h.arr<S>(buf, d);
            const hipError_t e = init_feq_device<S>(ptrs, c.l, c.m, c.n, h.nx, h.nxy, c.init, u00, h.stream);
            if (e != hipSuccess) return fail(BGK_EHIP, "device init failed: %s", hipGetErrorString(e));
        }
    } else if (c.init != 0) {
        return fail(BGK_EINVAL, "init mode %d not supported", c.init);
    }
    if (c.boundary == BGK_BC_INFLOW) {
        fill_inflow<S>(h);
        ENG_HIP(hipStreamSynchronize(h.stream));
    }
    return 0;
}

// Whether this handle's compact collide writes the inflow boundary's x
// faces itself (kFillsInflowFaces of the form it launches).
template <typename S>
bool collide_fills_faces(const bgk_handle& h)
{
    if (!h.compact || h.cfg.boundary != BGK_BC_INFLOW) return false;
    return h.cfg.les ? kFillsInflowFaces<S, 4> : kFillsInflowFaces<S, 0>;
}

// Rows for a call of `steps` steps of a handle that can have either.  Two steps
// per launch need padded rows and save about 0.7 of a step each time; a step
// alone takes 3 ... 23 % longer on them (us per step in calls of one step,
// compact against padded rows: FP32 130^3 60.4 / 68.5, 97 x 97 x 140 36.7 / 45.3,
// 200^3 204 / 223, 420 x 199 x 180 372 / 414; MIXED2 200^3 204 / 230; FP64 150^3 177 /
// 184).  The move takes about 1.5 steps, so it comes when the calls since the
// last one would have saved that much: before a long call at once, and back
// after some 15 calls of one step.
int choose_rows(bgk_handle& h, int steps)
{
    if (!h.flex || h.launch) return 0;
    const double saved = 0.7 * (steps / 2) - 0.1 * (steps % 2);
    h.owed = std::max(0.0, h.owed + (h.compact ? saved : -saved));
    if (h.owed < 1.5) return 0;
    h.owed = 0;
    return relayout(h, !h.compact);
}

// queue the boundary work and the fused collide of one step, or of two in
// one pass where that is faster and two are left, then swap; returns the
// steps taken.  `first`: the first launch of a stepping call, after which
// the lattice may have been set or restored -- the outflow kernel then runs
// whatever the collide writes.
template <typename S>
int one_launch(bgk_handle& h, int left, hipEvent_t pre, hipEvent_t post, bool first)
{
    const bool pair = h.pair && !h.compact && left >= 2;
    if (h.cfg.boundary == BGK_BC_INFLOW && (first || pair || !collide_fills_faces<S>(h))) {
        hipLaunchKernelGGL(outflow_halo<S>, dim3(ceil_div((long)h.cfg.m * h.cfg.n, 256)), dim3(256), 0, h.stream,
                           h.current<S>(), h.geom(), h.compact, (typename Storage<S>::compute)h.u_inflow);
    }
    if (pre) (void)hipEventRecord(pre, h.stream);
    launch_step<S>(h, pair);
    if (post) (void)hipEventRecord(post, h.stream);
    h.cur = 1 - h.cur;
    if (pair) h.rest = 1 - h.rest;
    h.steps += pair ? 2 : 1;
    return pair ? 2 : 1;
}

// Fortran sequential unformatted records: a 4-byte length, the data, the
// same length again (the layout amdflang and gfortran write for records
// below 2 GiB).
int write_record(FILE* f, const void* data, size_t bytes)
{
    const uint32_t len = (uint32_t)bytes;
    if (std::fwrite(&len, 4, 1, f) != 1 || (bytes && std::fwrite(data, 1, bytes, f) != bytes) ||
        std::fwrite(&len, 4, 1, f) != 1)
        return fail(BGK_EINVAL, "write error");
    return 0;
}

int read_record(FILE* f, void* data, size_t bytes, const char* path)
{
    uint32_t head = 0, tail = 0;
    if (std::fread(&head, 4, 1, f) != 1) return fail(BGK_EINVAL, "%s: truncated file", path);
    if (head != bytes)
        return fail(BGK_EINVAL, "%s: record of %u bytes, expected %zu (grid or storage type differ)", path, head,
                    bytes);
    if (std::fread(data, 1, bytes, f) != bytes || std::fread(&tail, 4, 1, f) != 1 || tail != head)
        return fail(BGK_EINVAL, "%s: damaged record", path);
    return 0;
}

template <typename S>
typename Storage<S>::compute cte_one()
{
    return typename Storage<S>::compute(1);
}

// The requested fields as FP64 arrays in host memory.  They are formed in the
// collision kind, so with FP32 half the bytes cross the bus; chunks of cells
// go through pinned memory, and a few threads, each with a chunk on its way,
// widen them into the caller's arrays.  What bounds it then is those arrays'
// first touch: 512 x 128^2 FP16 (268 MB) took 27 ms when FP64 copies to
// pageable memory did it all, 5.9 ms so (9.4 with the staging, at most 16 MB
// in FP32 and 32 MB in FP64, allocated on each call instead of kept by the
// handle).
template <typename S>
int download_fields(bgk_handle& h, double* const (&outs)[4])
{
    typedef typename Storage<S>::compute C;
    int want = 0, fields = 0;
    for (int q = 0; q < 4; ++q)
        if (outs[q]) want |= 1 << q, ++fields;
    if (!fields) return 0;
    const long cells = (long)h.cfg.l * h.cfg.m * h.cfg.n;
    const int chunk = (int)std::min(cells, std::max(1L << 15, std::min(1L << 17, cells / 8)));
    const int chunks = ceil_div(cells, chunk);
    const int cpus = std::max(1, (int)std::thread::hardware_concurrency());
    const int workers = std::min(chunks, std::min(8, cpus));
    const size_t slot = (size_t)chunk * fields;  // values of one chunk
    const size_t bytes = slot * workers * sizeof(C);
    // Threads may ask one handle for its fields at the same time: the staging
    // belongs to one of them until its copies are done.
    const std::lock_guard<std::mutex> lock(h.stage_lock);
    if (h.stage_bytes < bytes) {
        if (h.stage) (void)hipFree(h.stage);
        if (h.hstage) (void)hipHostFree(h.hstage);
        h.stage = h.hstage = nullptr;
        h.stage_bytes = 0;
        if (hipMalloc(&h.stage, bytes) != hipSuccess ||
            hipHostMalloc(&h.hstage, bytes, hipHostMallocDefault) != hipSuccess)
            return fail(BGK_ENOMEM, "fields staging");
        h.stage_bytes = bytes;
    }
    C *const dev = static_cast<C*>(h.stage), *const host = static_cast<C*>(h.hstage);
    std::atomic<int> next{0}, bad{0};
    auto work = [&](int w) {
        hipEvent_t done = nullptr;
        forget_error();
        bool ok = hipSetDevice(h.cfg.device) == hipSuccess &&
                  hipEventCreateWithFlags(&done, hipEventDisableTiming) == hipSuccess;
        C *d = dev + slot * w, *p = host + slot * w;
        for (int c; ok && !bad && (c = next++) < chunks;) {
            const long first = (long)c * chunk;
            const int count = (int)std::min<long>(chunk, cells - first);
            hipLaunchKernelGGL(fields_kernel<S>, dim3(ceil_div(count, 256)), dim3(256), 0, h.stream, h.current<S>(),
                               h.geom(), cte_one<S>(), first, count, want, d);
            ok = hipGetLastError() == hipSuccess &&
                 hipMemcpyAsync(p, d, (size_t)count * fields * sizeof(C), hipMemcpyDeviceToHost, h.stream) ==
                     hipSuccess &&
                 hipEventRecord(done, h.stream) == hipSuccess && hipEventSynchronize(done) == hipSuccess;
            const C* from = p;
            for (int q = 0; ok && q < 4; ++q) {
                if (!outs[q]) continue;
                double* to = outs[q] + first;
                for (int t = 0; t < count; ++t) to[t] = (double)from[t];
                from += count;
            }
        }
        if (!ok) bad = 1;
        if (done) (void)hipEventDestroy(done);
    };
    std::vector<std::thread> threads;
    try {
        threads.reserve(workers);
        for (int w = 1; w < workers; ++w) threads.emplace_back(work, w);
    } catch (...) {
        // no more threads to be had: those there are, and this one, do it all
    }
    work(0);
    for (std::thread& t : threads) t.join();
    int rc = bad ? fail(BGK_EHIP, "field download") : 0;
    if (hipStreamSynchronize(h.stream) != hipSuccess && rc == 0) rc = fail(BGK_EHIP, "fields");
    return rc;
}

}  // namespace

namespace bgk {
namespace eng {

int handle_setup(bgk_handle& h, const bgk_config& c, bool roomy)
{
    if (c.l < 1 || c.m < 1 || c.n < 1) return fail(BGK_EINVAL, "grid %d x %d x %d", c.l, c.m, c.n);
    if (c.boundary < 0 || c.boundary > 3) return fail(BGK_EINVAL, "boundary %d", c.boundary);
    if (c.storage < 0 || c.storage > 3) return fail(BGK_EINVAL, "storage %d", c.storage);
    if (c.init < 0 || c.init > 2) return fail(BGK_EINVAL, "init %d", c.init);
    if (c.obstacle < 0 || c.obstacle > 2) return fail(BGK_EINVAL, "obstacle %d", c.obstacle);
    if (c.obstacle && c.boundary != BGK_BC_INFLOW && c.boundary != BGK_BC_PERIODIC)
        return fail(BGK_EINVAL, "obstacles are supported with inflow or periodic boundaries");
    if (!(c.svisc > 0.0)) return fail(BGK_EINVAL, "svisc must be positive");
    if (c.force_axis < 1 || c.force_axis > 3) return fail(BGK_EINVAL, "force_axis %d", c.force_axis);
    if (c.wall_axis != 2 && c.wall_axis != 3) return fail(BGK_EINVAL, "wall_axis %d (2: y, 3: z)", c.wall_axis);
    if (c.boundary == BGK_BC_CHANNEL && c.wall_axis == 2 && c.force_axis == 2)
        return fail(BGK_EINVAL, "walls at y = 1, m: the body force must lie along them (force_axis 1 or 3)");
    if (c.les != 0 && c.les != 1) return fail(BGK_EINVAL, "les %d", c.les);
    if (c.mixed < 0 || c.mixed > 2) return fail(BGK_EINVAL, "mixed %d", c.mixed);
    if (c.mixed == 1 && c.storage != BGK_F16) return fail(BGK_EINVAL, "mixed 1 (MIXED1) stores FP16 (storage 2)");
    if (c.mixed == 2 && c.storage != BGK_F32) return fail(BGK_EINVAL, "mixed 2 (MIXED2) stores FP32 (storage 0)");
    if (c.obstacle) {
        // The link masks and the drag/lift mask cover the box centre +-
        // (radius + 4) clamped to the lattice, without wrapping: along a
        // periodic axis the box must lie inside, or cells across the seam
        // would pull from solid cells without bouncing back.
        const int ctr[3] = {c.obs_ic >= 0 ? c.obs_ic : 2 * c.l / 5, c.obs_jc >= 0 ? c.obs_jc : c.m / 2,
                            c.obs_kc >= 0 ? c.obs_kc : c.n / 2};
        const int R = c.obs_radius >= 0 ? c.obs_radius : (c.m > 256 ? 32 : c.m / 8);
        const int size[3] = {c.l, c.m, c.n};
        for (int ax = c.boundary == BGK_BC_PERIODIC ? 0 : 1; ax < 3; ++ax)
            if (ctr[ax] - (R + 4) < 1 || ctr[ax] + (R + 4) > size[ax])
                return fail(BGK_EINVAL,
                            "obstacle box %d +- %d leaves 1..%d along periodic axis %c: move the sphere away from "
                            "the seam",
                            ctr[ax], R + 4, size[ax], "xyz"[ax]);
    }
    if (c.layout < 0 || c.layout > 2) return fail(BGK_EINVAL, "layout %d", c.layout);
    h.cfg = c;
    h.esize = storage_bytes(c.storage);
    h.A = (int)(128 / h.esize);
    h.ny = c.m + 2;
    h.nz = c.n + 2;
    // Rows padded to whole lines, or compact rows where those measured
    // faster (prefer_compact: enough of a row's last line unused, or, with
    // 32/64-bit storage, a lattice of 2^24 cells or more).  Lattices that
    // take two steps per launch have padded rows: the tiles of collide_pair
    // start and end on lines (413 against 346 us per FP32 step at 256^3 over
    // compact rows).  They turn to compact rows where the caller takes one
    // step at a time (choose_rows).
    const double waste = (double)(round_up(c.l, h.A) - c.l) / (double)c.l;
    const bool compact = c.layout == 2 || (c.layout == 0 && prefer_compact(c, waste));
    h.pair = (roomy || !compact) && prefer_pair(c, round_up(c.l + 2, h.A) * h.ny, h.pgrid);
    h.flex = h.pair && compact;
    set_rows(h, compact && !h.pair);
    h.lstride = round_up(h.A + h.nxy * h.nz, h.A);
    // derived parameters in the collision kind (SRC/hencol.F90:31, :52;
    // SRC/bcond.driven.F90:61; SRC/build.bcond.F90:29-35)
    const bool dbl = compute_double(c);
    auto K = [&](double v) { return dbl ? v : (double)(float)v; };
    const double nu = K(c.svisc), u0f = K(c.boundary == BGK_BC_CHANNEL ? c.u0 : 0.0),
                 u00 = K(c.boundary == BGK_BC_CHANNEL ? 0.0 : c.u0);
    if (dbl) {
        h.omega = (1.0 + 1.0) / ((6.0 * nu) + 1.0);
        h.fgrad = 4.0 * u0f * nu / (5.0 * (double)c.m * (double)c.m);
        h.lidforce = u00 / 6.0;
    } else {
        const float nuf = (float)nu;
        h.omega = (1.0f + 1.0f) / ((6.0f * nuf) + 1.0f);
        h.fgrad = 4.0f * (float)u0f * nuf / (5.0f * (float)c.m * (float)c.m);
        h.lidforce = (float)u00 / 6.0f;
    }
    h.u_inflow = c.u_inflow < 0 ? (double)0.1f : K(c.u_inflow);
    h.cte_s = c.cte_s < 0 ? (double)0.1f : K(c.cte_s);

    return 0;
}

// Set up `h` where `free_bytes` of the device are free.  The padded rows of two
// steps per launch, up to 40 % more memory than compact rows, are taken only
// where the room they leave is at least eight times what they take beyond
// those, and 64 MB: what a program allocates next (the 8 bytes a cell of
// bgk_get_population; another handle) finds at least 8/9 of the room that it
// had beside compact rows.
static int setup_within(bgk_handle& h, const bgk_config& c, size_t free_bytes)
{
    if (int rc = handle_setup(h, c)) return rc;
    if (!h.flex) return 0;
    bgk_handle small;
    if (int rc = handle_setup(small, c, false)) return rc;
    const size_t padded = lattice_bytes(h), extra = padded - lattice_bytes(small);
    if (extra && free_bytes < padded + 8 * extra + (size_t(64) << 20)) return handle_setup(h, c, false);
    return 0;
}

int join_rest(bgk_handle& h)
{
    if (h.rest == h.cur) return 0;
    by_storage(h.cfg, [&](auto tag) {
        typedef decltype(tag) S;
        hipLaunchKernelGGL(move_rest<S>, dim3(ceil_div(h.plane * h.nz, 256)), dim3(256), 0, h.stream,
                           h.arr<S>(h.rest, 18), h.arr<S>(h.cur, 18), h.plane, h.nxy, h.nz);
        return 0;
    });
    h.rest = h.cur;
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? 0 : fail(BGK_EHIP, "direction 19: %s", hipGetErrorString(e));
}

// The populations go to the other lattice, the one they leave is cleared: a
// step's worth of reads and writes, and half of one more.
int relayout(bgk_handle& h, bool compact)
{
    if (h.compact == compact) return 0;
    if (int rc = join_rest(h)) return rc;
    return by_storage(h.cfg, [&](auto tag) {
        typedef decltype(tag) S;
        const Lattice19<S> from = h.current<S>();
        const Geometry gf = h.geom();
        const int left = h.cur;
        h.cur = h.rest = 1 - left;
        set_rows(h, compact);
        hipLaunchKernelGGL(move_rows<S>, dim3(ceil_div(h.plane * h.nz, 256)), dim3(256), 0, h.stream, from, gf,
                           h.current<S>(), h.geom(), h.plane);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail(BGK_EHIP, "rows: %s", hipGetErrorString(e));
        ENG_HIP(hipMemsetAsync(h.mem[left], 0, (size_t)h.lstride * h.esize, h.stream));
        if (h.cfg.boundary == BGK_BC_INFLOW) fill_inflow<S>(h);
        return 0;
    });
}

}  // namespace eng
}  // namespace bgk

extern "C" {

void bgk_config_default(bgk_config* c, int l, int m, int n)
{
    std::memset(c, 0, sizeof *c);
    c->l = l;
    c->m = m;
    c->n = n;
    c->boundary = BGK_BC_DRIVEN;
    c->storage = BGK_F32;
    c->svisc = 0.064;
    c->u0 = 0.1;
    c->obs_ic = c->obs_jc = c->obs_kc = c->obs_radius = -1;
    c->u_inflow = -1.0;
    c->force_axis = 1;
    c->les = 0;
    c->cte_s = -1.0;
    c->wall_axis = 3;
    c->mixed = 0;
    c->layout = 0;
}

const char* bgk_last_error(void) { return last_error(); }

int bgk_plan(const bgk_config* cfg, size_t free_bytes, long long out[5])
{
    if (!cfg || !out) return fail(BGK_EINVAL, "null argument");
    bgk_handle h;
    if (int rc = setup_within(h, *cfg, free_bytes)) return rc;
    out[0] = h.pair ? 2 : 1;
    out[1] = h.compact;
    out[2] = (long long)lattice_bytes(h);
    out[3] = h.pair ? h.pgrid.th : 0;
    out[4] = h.pair ? h.pgrid.zc : 0;
    return 0;
}

int bgk_create(const bgk_config* cfg, bgk_handle** out)
{
    if (!cfg || !out) return fail(BGK_EINVAL, "null argument");
    *out = nullptr;
    const bgk_config& c = *cfg;
    bgk_handle* h = new bgk_handle();
    if (int rc = handle_setup(*h, c)) {
        delete h;
        return rc;
    }
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || c.device < 0 || c.device >= ndev) {
        delete h;
        return fail(BGK_EINVAL, "device %d not available (%d devices)", c.device, ndev);
    }
    if (hipSetDevice(c.device) != hipSuccess) {
        delete h;
        return fail(BGK_EHIP, "hipSetDevice(%d) failed", c.device);
    }
    forget_error();
    size_t free_bytes = 0, total = 0;
    if (h->flex && hipMemGetInfo(&free_bytes, &total) == hipSuccess) (void)setup_within(*h, c, free_bytes);

    int rc = 0;
    auto cleanup = [&](int code) {
        bgk_destroy(h);
        return code;
    };
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(fail(BGK_EHIP, "stream creation failed"));
    void* region = nullptr;
    hipError_t got = hipMalloc(&region, lattice_bytes(*h));
    if (got != hipSuccess && h->pair) {  // padded rows do not fit: compact ones may
        forget_error();
        handle_setup(*h, c, false);
        got = hipMalloc(&region, lattice_bytes(*h));
    }
    if (got != hipSuccess)
        return cleanup(fail(BGK_ENOMEM, "cannot allocate %.2f GB of lattice", lattice_bytes(*h) / 1e9));
    place_lattices(*h, region);
    if (hipMemsetAsync(region, 0, lattice_bytes(*h), h->stream) != hipSuccess)
        return cleanup(fail(BGK_EHIP, "lattice clear failed"));

    // obstacle: reference sphere shell by default (SRC/build.obs.F90:52-60)
    if (c.obstacle) {
        h->has_obs = true;
        h->ic = c.obs_ic >= 0 ? c.obs_ic : 2 * c.l / 5;
        h->jc = c.obs_jc >= 0 ? c.obs_jc : c.m / 2;
        h->kc = c.obs_kc >= 0 ? c.obs_kc : c.n / 2;
        h->radius = c.obs_radius >= 0 ? c.obs_radius : (c.m > 256 ? 32 : c.m / 8);
        const int R = h->radius + 3;
        // link masks for every cell within R+1 of the centre (bit d: x - c_d solid)
        int lo[3] = {std::max(1, h->ic - R), std::max(1, h->jc - R), std::max(1, h->kc - R)};
        int hi[3] = {std::min(c.l, h->ic + R), std::min(c.m, h->jc + R), std::min(c.n, h->kc + R)};
        const int ni = hi[0] - lo[0] + 1, nj = hi[1] - lo[1] + 1, nk = hi[2] - lo[2] + 1;
        std::vector<uint32_t> bits((size_t)ni * nj * nk, 0u);
        const bool px = c.boundary == BGK_BC_PERIODIC;
        for (int k = lo[2]; k <= hi[2]; ++k)
            for (int j = lo[1]; j <= hi[1]; ++j)
                for (int i = lo[0]; i <= hi[0]; ++i) {
                    uint32_t b = 0;
                    for (int d = 0; d < 18; ++d) {
                        int si = i - cx_of(d), sj = wrap(j - cy_of(d), c.m), sk = wrap(k - cz_of(d), c.n);
                        if (px) si = wrap(si, c.l);
                        if (sphere_solid(*h, si, sj, sk)) b |= 1u << d;
                    }
                    bits[(size_t)(i - lo[0]) + (size_t)ni * ((j - lo[1]) + (size_t)nj * (k - lo[2]))] = b;
                }
        h->ob[0] = lo[0];
        h->ob[1] = lo[1];
        h->ob[2] = lo[2];
        h->ob[3] = ni;
        h->ob[4] = nj;
        h->ob[5] = nk;
        // solid mask over centre +- (radius + 4) for the drag/lift sums
        const int Q = h->radius + 4;
        int mlo[3] = {std::max(1, h->ic - Q), std::max(1, h->jc - Q), std::max(1, h->kc - Q)};
        int mhi[3] = {std::min(c.l, h->ic + Q), std::min(c.m, h->jc + Q), std::min(c.n, h->kc + Q)};
        const int mi = mhi[0] - mlo[0] + 1, mj = mhi[1] - mlo[1] + 1, mkk = mhi[2] - mlo[2] + 1;
        std::vector<int8_t> mask((size_t)mi * mj * mkk, 0);
        for (int k = mlo[2]; k <= mhi[2]; ++k)
            for (int j = mlo[1]; j <= mhi[1]; ++j)
                for (int i = mlo[0]; i <= mhi[0]; ++i)
                    mask[(size_t)(i - mlo[0]) + (size_t)mi * ((j - mlo[1]) + (size_t)mj * (k - mlo[2]))] =
                        sphere_solid(*h, i, j, k) ? 1 : 0;
        h->mk[0] = mlo[0];
        h->mk[1] = mlo[1];
        h->mk[2] = mlo[2];
        h->mk[3] = mi;
        h->mk[4] = mj;
        h->mk[5] = mkk;
        if (hipMalloc(&h->obits, bits.size() * 4) != hipSuccess || hipMalloc(&h->omask, mask.size()) != hipSuccess)
            return cleanup(fail(BGK_ENOMEM, "obstacle masks"));
        if (hipMemcpy(h->obits, bits.data(), bits.size() * 4, hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(h->omask, mask.data(), mask.size(), hipMemcpyHostToDevice) != hipSuccess)
            return cleanup(fail(BGK_EHIP, "obstacle upload"));
    }
    if (hipMalloc(&h->scratch, (kRedBlocks + 8) * 5 * sizeof(double)) != hipSuccess ||
        hipHostMalloc(&h->hscratch, (kRedBlocks + 8) * 5 * sizeof(double), hipHostMallocDefault) != hipSuccess)
        return cleanup(fail(BGK_ENOMEM, "scratch"));
    if (hipStreamSynchronize(h->stream) != hipSuccess) return cleanup(fail(BGK_EHIP, "memset"));
    rc = by_storage(c, [&](auto tag) { return upload_state<decltype(tag)>(*h); });
    if (rc) return cleanup(rc);
    *out = h;
    return 0;
}

int bgk_destroy(bgk_handle* h)
{
    if (!h) return 0;
    if (h->stream) (void)hipStreamSynchronize(h->stream);
    for (auto e : h->events) (void)hipEventDestroy(e);
    if (h->obits) (void)hipFree(h->obits);
    if (h->omask) (void)hipFree(h->omask);
    if (h->stage) (void)hipFree(h->stage);
    if (h->hstage) (void)hipHostFree(h->hstage);
    if (!h->borrowed) {
        if (h->mem[0]) (void)hipFree(h->mem[0]);  // one region holds both lattices
        if (h->scratch) (void)hipFree(h->scratch);
        if (h->hscratch) (void)hipHostFree(h->hscratch);
        if (h->stream) (void)hipStreamDestroy(h->stream);
    }
    delete h;
    return 0;
}

int bgk_step(bgk_handle* h, int nsteps)
{
    if (!h || nsteps < 0) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    forget_error();
    if (int rc = choose_rows(*h, nsteps)) return rc;
    return by_storage(h->cfg, [&](auto tag) {
        for (int s = 0; s < nsteps;) s += one_launch<decltype(tag)>(*h, nsteps - s, nullptr, nullptr, s == 0);
        hipError_t e = hipGetLastError();
        return e == hipSuccess ? 0 : fail(BGK_EHIP, "step launch: %s", hipGetErrorString(e));
    });
}

int bgk_sync(bgk_handle* h)
{
    if (!h) return fail(BGK_EINVAL, "null handle");
    ENG_HIP(hipStreamSynchronize(h->stream));
    return 0;
}

int bgk_time_steps(bgk_handle* h, int nsteps, double* total_ms, double* collide_avg_ms)
{
    if (!h || nsteps < 1) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const size_t need = 2 * (size_t)nsteps + 2;
    while (h->events.size() < need) {
        hipEvent_t e;
        ENG_HIP(hipEventCreate(&e));
        h->events.push_back(e);
    }
    ENG_HIP(hipStreamSynchronize(h->stream));
    forget_error();
    hipEvent_t e0 = h->events[0], e1 = h->events[1];
    ENG_HIP(hipEventRecord(e0, h->stream));
    if (int rc = choose_rows(*h, nsteps)) return rc;
    int launches = 0;
    int rc = by_storage(h->cfg, [&](auto tag) {
        for (int s = 0; s < nsteps; ++launches)
            s += one_launch<decltype(tag)>(*h, nsteps - s, h->events[2 + 2 * launches], h->events[3 + 2 * launches],
                                           s == 0);
        return 0;
    });
    if (rc) return rc;
    ENG_HIP(hipEventRecord(e1, h->stream));
    ENG_HIP(hipEventSynchronize(e1));
    float ms = 0;
    ENG_HIP(hipEventElapsedTime(&ms, e0, e1));
    double ksum = 0;
    for (int s = 0; s < launches; ++s) {
        float k = 0;
        ENG_HIP(hipEventElapsedTime(&k, h->events[2 + 2 * s], h->events[3 + 2 * s]));
        ksum += k;
    }
    if (total_ms) *total_ms = ms;
    if (collide_avg_ms) *collide_avg_ms = ksum / nsteps;
    return 0;
}

int bgk_diagno(bgk_handle* h, double out[5])
{
    if (!h || !out) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const DiagnoGrid dg = diagno_grid(h->cfg.l, (long)h->cfg.m * h->cfg.n);
    int rc = by_storage(h->cfg, [&](auto tag) {
        typedef decltype(tag) S;
        launch_diagno(h->current<S>(), h->geom(), cte_one<S>(), dg, h->scratch, h->stream);
        hipLaunchKernelGGL(fold_partials<5>, dim3(1), dim3(kRedThreads), 0, h->stream, h->scratch, dg.blocks,
                           h->hscratch);
        return 0;
    });
    if (rc) return rc;
    ENG_HIP(hipStreamSynchronize(h->stream));
    const double fl = (double)(float)h->cfg.l, fm = (double)(float)h->cfg.m, fn = (double)(float)h->cfg.n;
    for (int q = 0; q < 5; ++q) out[q] = (h->hscratch[q] / fl) / fm / fn;
    return 0;
}

int bgk_draglift(bgk_handle* h, double out[3])
{
    if (!h || !out) return fail(BGK_EINVAL, "bad arguments");
    if (!h->has_obs) return fail(BGK_EINVAL, "no obstacle");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const bgk_config& c = h->cfg;
    const int delta = 3;  // SRC/draglift.F90:54
    const int is = std::max(1, h->ic - h->radius - delta), ie = std::min(c.l, h->ic + h->radius + delta);
    const int js = std::max(1, h->jc - h->radius - delta), je = std::min(c.m, h->jc + h->radius + delta);
    const int ks = std::max(1, h->kc - h->radius - delta), ke = std::min(c.n, h->kc + h->radius + delta);
    const long cells = (long)(ie - is + 1) * (je - js + 1) * (ke - ks + 1);
    const int nb = (int)std::min<long>((cells + kRedThreads - 1) / kRedThreads, kRedBlocks);
    by_storage(c, [&](auto tag) {
        typedef decltype(tag) S;
        hipLaunchKernelGGL(draglift_box<S>, dim3(nb), dim3(kRedThreads), 0, h->stream, h->current<S>(), h->geom(),
                           h->omask, h->mk[0], h->mk[1], h->mk[2], h->mk[3], h->mk[4], h->mk[5], is, ie, js, je, ks,
                           ke, h->scratch);
        hipLaunchKernelGGL(fold_partials<3>, dim3(1), dim3(kRedThreads), 0, h->stream, h->scratch, nb, h->hscratch);
        return 0;
    });
    ENG_HIP(hipStreamSynchronize(h->stream));
    // norm = uno/(u_inflow*u_inflow*radius) in the working kind (SRC/draglift.F90:178)
    double norm;
    if (compute_double(c))
        norm = 1.0 / (h->u_inflow * h->u_inflow * (double)h->radius);
    else {
        const float u = (float)h->u_inflow;
        norm = (double)(1.0f / (u * u * (float)h->radius));
    }
    for (int q = 0; q < 3; ++q) out[q] = h->hscratch[q] * norm;
    return 0;
}

int bgk_fields(bgk_handle* h, double* rho, double* ux, double* uy, double* uz)
{
    if (!h) return fail(BGK_EINVAL, "null handle");
    ENG_HIP(hipSetDevice(h->cfg.device));
    double* const outs[4] = {rho, ux, uy, uz};
    return by_storage(h->cfg, [&](auto tag) { return download_fields<decltype(tag)>(*h, outs); });
}

int bgk_profile(bgk_handle* h, int axis, int c1, int c2, double* out)
{
    if (!h || !out || axis < 0 || axis > 2) return fail(BGK_EINVAL, "bad arguments");
    const bgk_config& c = h->cfg;
    const int len = axis == 0 ? c.l : (axis == 1 ? c.m : c.n);
    const int lim1 = axis == 0 ? c.m : c.l, lim2 = axis == 2 ? c.m : c.n;
    if (c1 < 1 || c1 > lim1 || c2 < 1 || c2 > lim2)
        return fail(BGK_EINVAL, "line (%d,%d) outside the interior", c1, c2);
    ENG_HIP(hipSetDevice(c.device));
    return by_storage(c, [&](auto tag) {
        typedef decltype(tag) S;
        typedef typename Storage<S>::compute C;
        C* tmp = nullptr;
        if (hipMalloc(&tmp, (size_t)4 * len * sizeof(C)) != hipSuccess) return fail(BGK_ENOMEM, "profile");
        hipLaunchKernelGGL(prof_line_kernel<S>, dim3(ceil_div(len, 64)), dim3(64), 0, h->stream, h->current<S>(),
                           h->geom(), axis, c1, c2, 1, len, cte_one<S>(), tmp);
        std::vector<C> host((size_t)4 * len);
        int r = 0;
        if (hipMemcpyAsync(host.data(), tmp, host.size() * sizeof(C), hipMemcpyDeviceToHost, h->stream) !=
                hipSuccess ||
            hipStreamSynchronize(h->stream) != hipSuccess)
            r = fail(BGK_EHIP, "profile download");
        for (size_t q = 0; q < host.size(); ++q) out[q] = (double)host[q];
        (void)hipFree(tmp);
        return r;
    });
}

int bgk_prof_k(bgk_handle* h, int icoord, int jcoord, double* out) { return bgk_profile(h, 2, icoord, jcoord, out); }

int bgk_probe(bgk_handle* h, int i0, int j0, int k0, double out[4])
{
    if (!h || !out) return fail(BGK_EINVAL, "bad arguments");
    const bgk_config& c = h->cfg;
    if (i0 < 1 || i0 > c.l || j0 < 1 || j0 > c.m || k0 < 1 || k0 > c.n)
        return fail(BGK_EINVAL, "point (%d,%d,%d) outside the interior", i0, j0, k0);
    ENG_HIP(hipSetDevice(c.device));
    return by_storage(c, [&](auto tag) {
        typedef decltype(tag) S;
        typedef typename Storage<S>::compute C;
        C* tmp = nullptr;
        if (hipMalloc(&tmp, 4 * sizeof(C)) != hipSuccess) return fail(BGK_ENOMEM, "probe");
        hipLaunchKernelGGL(prof_line_kernel<S>, dim3(1), dim3(64), 0, h->stream, h->current<S>(), h->geom(), 0, j0,
                           k0, i0, 1, cte_one<S>(), tmp);
        C host[4];
        int r = 0;
        if (hipMemcpyAsync(host, tmp, sizeof host, hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
            hipStreamSynchronize(h->stream) != hipSuccess)
            r = fail(BGK_EHIP, "probe download");
        for (int q = 0; q < 4; ++q) out[q] = (double)host[q];
        (void)hipFree(tmp);
        return r;
    });
}

int bgk_get_population(bgk_handle* h, int dir, double* out)
{
    if (!h || !out || dir < 0 || dir > 18) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const long cells = (long)h->cfg.l * h->cfg.m * h->cfg.n;
    double* d = nullptr;
    ENG_HIP(hipMalloc(&d, cells * sizeof(double)));
    by_storage(h->cfg, [&](auto tag) {
        typedef decltype(tag) S;
        hipLaunchKernelGGL(get_interior<S>, dim3(ceil_div(cells, 256)), dim3(256), 0, h->stream, h->cur_a<S>(dir),
                           h->geom(), d);
        return 0;
    });
    int rc = 0;
    if (hipMemcpyAsync(out, d, cells * sizeof(double), hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
        hipStreamSynchronize(h->stream) != hipSuccess)
        rc = fail(BGK_EHIP, "population download");
    (void)hipFree(d);
    return rc;
}

int bgk_set_population(bgk_handle* h, int dir, const double* in)
{
    if (!h || !in || dir < 0 || dir > 18) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const long cells = (long)h->cfg.l * h->cfg.m * h->cfg.n;
    double* d = nullptr;
    ENG_HIP(hipMalloc(&d, cells * sizeof(double)));
    int rc = 0;
    if (hipMemcpyAsync(d, in, cells * sizeof(double), hipMemcpyHostToDevice, h->stream) != hipSuccess)
        rc = fail(BGK_EHIP, "population upload");
    if (rc == 0)
        by_storage(h->cfg, [&](auto tag) {
            typedef decltype(tag) S;
            hipLaunchKernelGGL(set_interior<S>, dim3(ceil_div(cells, 256)), dim3(256), 0, h->stream, h->cur_a<S>(dir),
                               h->geom(), d);
            return 0;
        });
    if (hipStreamSynchronize(h->stream) != hipSuccess && rc == 0) rc = fail(BGK_EHIP, "population set");
    (void)hipFree(d);
    return rc;
}

// ---- on-disk formats -------------------------------------------------------

int bgk_save_raw(bgk_handle* h, const char* path, int itime)
{
    if (!h || !path) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const bgk_config& c = h->cfg;
    const long cnt = (long)(c.l + 2) * (c.m + 2) * (c.n + 2);
    const size_t bytes = (size_t)cnt * h->esize;
    if (bytes > 0x7fffffffu) return fail(BGK_EINVAL, "record of %zu bytes does not fit a 4-byte record marker", bytes);
    FILE* f = std::fopen(path, "wb");
    if (!f) return fail(BGK_EINVAL, "cannot open %s for writing", path);
    void* dev = nullptr;
    std::vector<char> host(bytes);
    int rc = hipMalloc(&dev, bytes) == hipSuccess ? 0 : fail(BGK_ENOMEM, "save_raw staging");
    if (rc == 0) rc = write_record(f, &itime, 4);
    for (int d = 0; d < 19 && rc == 0; ++d) {
        rc = by_storage(c, [&](auto tag) {
            typedef decltype(tag) S;
            hipLaunchKernelGGL(pack_halo<S>, dim3(ceil_div(cnt, 256)), dim3(256), 0, h->stream, h->cur_a<S>(d),
                               h->geom(), static_cast<S*>(dev));
            return 0;
        });
        if (rc == 0 && (hipMemcpyAsync(host.data(), dev, bytes, hipMemcpyDeviceToHost, h->stream) != hipSuccess ||
                        hipStreamSynchronize(h->stream) != hipSuccess))
            rc = fail(BGK_EHIP, "save_raw download");
        if (rc == 0) rc = write_record(f, host.data(), bytes);
    }
    if (dev) (void)hipFree(dev);
    if (std::fclose(f) != 0 && rc == 0) rc = fail(BGK_EINVAL, "write error on %s", path);
    return rc;
}

int bgk_restore_raw(bgk_handle* h, const char* path, int* itime)
{
    if (!h || !path) return fail(BGK_EINVAL, "bad arguments");
    ENG_HIP(hipSetDevice(h->cfg.device));
    const bgk_config& c = h->cfg;
    const long cnt = (long)(c.l + 2) * (c.m + 2) * (c.n + 2);
    const size_t bytes = (size_t)cnt * h->esize;
    FILE* f = std::fopen(path, "rb");
    if (!f) return fail(BGK_EINVAL, "cannot open %s", path);
    int it = 0;
    void* dev = nullptr;
    std::vector<char> host(bytes);
    int rc = read_record(f, &it, 4, path);
    if (rc == 0 && hipMalloc(&dev, bytes) != hipSuccess) rc = fail(BGK_ENOMEM, "restore_raw staging");
    for (int d = 0; d < 19 && rc == 0; ++d) {
        rc = read_record(f, host.data(), bytes, path);
        if (rc) break;
        if (hipMemcpyAsync(dev, host.data(), bytes, hipMemcpyHostToDevice, h->stream) != hipSuccess) {
            rc = fail(BGK_EHIP, "restore_raw upload");
            break;
        }
        rc = by_storage(c, [&](auto tag) {
            typedef decltype(tag) S;
            hipLaunchKernelGGL(unpack_halo<S>, dim3(ceil_div(cnt, 256)), dim3(256), 0, h->stream,
                               static_cast<const S*>(dev), h->geom(), h->cur_a<S>(d));
            return 0;
        });
        if (rc == 0 && hipStreamSynchronize(h->stream) != hipSuccess) rc = fail(BGK_EHIP, "restore_raw");
    }
    std::fclose(f);
    if (dev) (void)hipFree(dev);
    if (rc) return rc;
    // the engine's own constant inflow face (both lattices)
    if (c.boundary == BGK_BC_INFLOW) {
        rc = by_storage(c, [&](auto tag) {
            fill_inflow<decltype(tag)>(*h);
            return hipStreamSynchronize(h->stream) == hipSuccess ? 0 : fail(BGK_EHIP, "inflow face");
        });
        if (rc) return rc;
    }
    h->steps = it;
    if (itime) *itime = it;
    return 0;
}

int bgk_save_vel(bgk_handle* h, const char* path, int itime)
{
    if (!h || !path) return fail(BGK_EINVAL, "bad arguments");
    const bgk_config& c = h->cfg;
    const long cells = (long)c.l * c.m * c.n;
    std::vector<double> ux(cells), uy(cells), uz(cells);
    if (int rc = bgk_fields(h, nullptr, ux.data(), uy.data(), uz.data())) return rc;
    FILE* f = std::fopen(path, "wb");
    if (!f) return fail(BGK_EINVAL, "cannot open %s for writing", path);
    int rc = write_record(f, &itime, 4);
    // one record per cell, three values of the collision kind (i fastest)
    for (long t = 0; t < cells && rc == 0; ++t) {
        if (compute_double(c)) {
            const double v[3] = {ux[t], uy[t], uz[t]};
            rc = write_record(f, v, sizeof v);
        } else {
            const float v[3] = {(float)ux[t], (float)uy[t], (float)uz[t]};
            rc = write_record(f, v, sizeof v);
        }
    }
    if (std::fclose(f) != 0 && rc == 0) rc = fail(BGK_EINVAL, "write error on %s", path);
    return rc;
}

int bgk_write_vtk(bgk_handle* h, int kind, int index, const char* path)
{
    if (!h || !path || kind < 0 || kind > 3) return fail(BGK_EINVAL, "bad arguments");
    const bgk_config& c = h->cfg;
    const int lim = kind == 0 || kind == 3 ? c.n : (kind == 1 ? c.m : c.l);
    if (index < 1 || index > lim) return fail(BGK_EINVAL, "plane index %d outside 1..%d", index, lim);
    if (kind == 3 && (c.l < 3 || c.m < 3 || index < 2 || index > c.n - 1))
        return fail(BGK_EINVAL, "vorticity plane needs l, m >= 3 and 2 <= k0 <= n-1");
    ENG_HIP(hipSetDevice(c.device));
    int dims[3], origin[3];
    long npts;
    const char* vec = " VECTORS velocity float";
    switch (kind) {
        case 0: dims[0] = c.l, dims[1] = c.m, dims[2] = 1, origin[0] = 1, origin[1] = 1, origin[2] = index; break;
        case 1: dims[0] = c.l, dims[1] = 1, dims[2] = c.n, origin[0] = 1, origin[1] = index, origin[2] = 1; break;
        case 2: dims[0] = 1, dims[1] = c.m, dims[2] = c.n, origin[0] = index, origin[1] = 1, origin[2] = 1; break;
        default:
            dims[0] = c.l - 2, dims[1] = c.m - 2, dims[2] = 1, origin[0] = 2, origin[1] = 2, origin[2] = index;
            vec = " VECTORS vorticity float";
    }
    npts = (long)dims[0] * dims[1] * dims[2];
    float* dev = nullptr;
    ENG_HIP(hipMalloc(&dev, (size_t)npts * 3 * sizeof(float)));
    by_storage(c, [&](auto tag) {
        typedef decltype(tag) S;
        if (kind == 3)
            hipLaunchKernelGGL(vorticity_xy_kernel<S>, dim3(ceil_div(npts, 256)), dim3(256), 0, h->stream,
                               h->current<S>(), h->geom(), index, dev);
        else
            hipLaunchKernelGGL(vtk_plane_kernel<S>, dim3(ceil_div(npts, 256)), dim3(256), 0, h->stream,
                               h->current<S>(), h->geom(), kind, index, dev);
        return 0;
    });
    std::vector<float> host((size_t)npts * 3);
    int rc = 0;
    if (hipMemcpyAsync(host.data(), dev, host.size() * sizeof(float), hipMemcpyDeviceToHost, h->stream) !=
            hipSuccess ||
        hipStreamSynchronize(h->stream) != hipSuccess)
        rc = fail(BGK_EHIP, "vtk download");
    (void)hipFree(dev);
    if (rc) return rc;
    // ASCII header as the reference's formatted writes produce it
    // (SRC/vtk_xy.binary.F90:61-72: A10 cuts 'POINT_DATA ' to 10
    // characters, A23/A24 right-justify the VECTORS line), then big-endian
    // FP32 triplets.
    char head[512];
    const int len = std::snprintf(head, sizeof head,
                                  "# vtk DataFile Version 2.0\nCampo\nBINARY\nDATASET STRUCTURED_POINTS\n"
                                  "DIMENSIONS %10d %10d %10d\nORIGIN %10d %10d %10d\nSPACING %10d %10d %10d\n"
                                  "POINT_DATA%10ld\n%s\n",
                                  dims[0], dims[1], dims[2], origin[0], origin[1], origin[2], 1, 1, 1, npts, vec);
    for (float& v : host) {
        uint32_t u;
        std::memcpy(&u, &v, 4);
        u = __builtin_bswap32(u);
        std::memcpy(&v, &u, 4);
    }
    FILE* f = std::fopen(path, "wb");
    if (!f) return fail(BGK_EINVAL, "cannot open %s for writing", path);
    if (std::fwrite(head, 1, (size_t)len, f) != (size_t)len ||
        std::fwrite(host.data(), sizeof(float), host.size(), f) != host.size())
        rc = fail(BGK_EINVAL, "write error on %s", path);
    if (std::fclose(f) != 0 && rc == 0) rc = fail(BGK_EINVAL, "write error on %s", path);
    return rc;
}

int bgk_info(bgk_handle* h, long long out[6])
{
    if (!h || !out) return fail(BGK_EINVAL, "bad arguments");
    out[0] = h->nx;
    out[1] = h->ny;
    out[2] = h->nz;
    out[3] = (long long)h->bytes;
    out[4] = (long long)h->esize;
    out[5] = h->steps;
    return 0;
}

int bgk_set_launch(bgk_handle* h, int steps, int rows, int planes)
{
    if (!h || steps < 0 || steps > 2 || rows < 0 || planes < 0) return fail(BGK_EINVAL, "bad arguments");
    const bgk_config& c = h->cfg;
    const bool padded = h->flex || !h->compact;
    const long plane = round_up(c.l + 2, h->A) * h->ny;
    PairGrid g{};
    const bool rule = padded && prefer_pair(c, plane, g);
    if (steps == 2) {
        if (!padded || !can_pair(c, plane))
            return fail(BGK_EINVAL, "two steps per launch need FP32 or FP64 storage on padded rows (layout 1)");
        if (rows > pair_rows_max(c) || planes > c.n)
            return fail(BGK_EINVAL, "tiles of %d rows, %d planes: at most %d and %d", rows, planes, pair_rows_max(c),
                        c.n);
        if (rows || planes) g = pair_grid_of(c.l, c.m, c.n, rows ? rows : g.th, planes ? planes : g.zc);
        if (g.total <= 0) return fail(BGK_EINVAL, "more than 2^30 tiles");
    } else if (rows || planes) {
        return fail(BGK_EINVAL, "tiles are those of two steps per launch");
    }
    ENG_HIP(hipSetDevice(c.device));
    forget_error();
    if (steps && h->flex)
        if (int rc = relayout(*h, steps == 1)) return rc;
    h->launch = steps;
    h->pair = steps ? steps == 2 : rule;
    h->pgrid = g;
    return 0;
}

int bgk_launch_info(bgk_handle* h, long long out[4])
{
    if (!h || !out) return fail(BGK_EINVAL, "bad arguments");
    out[0] = h->pair ? 2 : 1;
    out[1] = h->compact;
    out[2] = h->pair ? h->pgrid.th : 0;
    out[3] = h->pair ? h->pgrid.zc : 0;
    return 0;
}

}  // extern "C"
