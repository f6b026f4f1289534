"""The work a user of this framework has it do, as timed cases.

Three ways into the framework:

* ``engine``: a handle of the library's own lattices (``Engine``).  A pass
  runs one output interval -- ``steps`` time steps, then the macroscopic
  fields -- and returns density and velocity.  Runs of this kind take
  thousands of steps between outputs (the stored cases check every 1000 to
  20000 steps), so the steps are most of a pass here too.
* ``v1``: the reference-compatible ABI on the caller's arrays
  (``Simulation``): per step the boundary routine, ``col_mc_gpu`` and the
  pointer swap.  A pass runs ``steps`` steps and returns the interior of the
  19 population arrays.
* ``diag``: that ABI's reductions on a developed state, the set the
  reference prints at every check: means, plane means, the three line
  profiles, a probe and the obstacle's drag.
* ``serve``: the batching server.  A pass submits a mix of cavity requests,
  advances the server until all are done and returns their diagnostics.

The viscosity and the driving velocity of a case come from the seed (within
10 % of the case's own), so two seeds are two flows.
"""
import math
import random

import numpy as np
import torch

from bgk3d_gpu_amd.cases import Case, sphere_obstacle
from bgk3d_gpu_amd.engine import Engine
from bgk3d_gpu_amd.serving import Request, Server
from bgk3d_gpu_amd.simulation import Simulation

BYTES = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2}


def _engine(name, boundary, l, m, n, storage, steps, **kw):
    c = dict(kind="engine", boundary=boundary, l=l, m=m, n=n, storage=storage, steps=steps, rounding=0, mixed=0,
             les=False, wall_axis=3, obstacle=False, nu=0.02, u0=0.1, before=0)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def _v1(name, boundary, l, m, n, prec, steps, **kw):
    c = dict(kind="v1", boundary=boundary, l=l, m=m, n=n, prec=prec, steps=steps, les=False, obstacle=False, nu=0.02,
             u0=0.1)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest problem in the configurations: the 64^3 cavity at Re = 100 with its 2000 steps, where a step
        # is a launch and little else
        _engine("cavity_64_f32", "ldc", 64, 64, 64, "f32", 2000, nu=0.064),
        # the benchmark's flow and size, between two outputs
        _engine("taylor_green_256_f32", "periodic", 256, 256, 256, "f32", 500, nu=0.01, u0=0.05),
        # the same flow in double precision
        _engine("taylor_green_192_f64", "periodic", 192, 192, 192, "f64", 300, nu=0.01, u0=0.05),
        # body-force channel of the precision study, FP16 with stochastic rounding, walls in y
        _engine("channel_512x128x128_f16", "channel", 512, 128, 128, "f16", 500, rounding=1, wall_axis=2, nu=0.1,
                u0=0.02048),
        # a served size that fits no tile, in BF16
        _engine("cavity_149_bf16", "ldc", 149, 149, 149, "bf16", 600, rounding=1, nu=0.05),
        # flow past the sphere shell at the stored input's size, once the start-up wave has met the sphere
        _engine("sphere_900x150x150_f32", "inflow", 900, 150, 150, "f32", 200, obstacle=True, nu=0.01, before=500),
        # large-eddy run, odd sizes
        _engine("les_201x135x99_f32", "periodic", 201, 135, 99, "f32", 800, les=True, nu=0.001, u0=0.05),
        # the caller's own arrays: a small cavity in double precision, where the calls themselves count
        _v1("abi_cavity_64_f64", "ldc", 64, 64, 64, "dp", 100, nu=0.064),
        # the caller's arrays at the benchmark's size
        _v1("abi_taylor_green_256_f32", "periodic", 256, 256, 256, "sp", 20, nu=0.01, u0=0.05),
        # the largest lattice of the stored inputs
        _v1("abi_taylor_green_400_f32", "periodic", 400, 400, 400, "sp", 10, nu=0.004, u0=0.05),
        # what is printed at every check of the sphere run
        dict(name="abi_diagnostics_450x150x150_f32", kind="diag", boundary="inflow", l=450, m=150, n=150, prec="sp",
             steps=8, les=False, obstacle=True, nu=0.01, u0=0.1),
        # a sweep of cavities served from one process
        dict(name="serve_8_cavities", kind="serve", count=8, n_lo=32, n_hi=160, steps=1000, mix=0),
    ]


def _size(rng, lo, hi):
    """Log-uniform size, odd ones among them."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["engine"] * 6 + ["v1"] * 3 + ["diag", "serve"])
    if kind == "serve":
        lo = rng.randint(32, 64)
        return dict(kind="serve", count=rng.randint(3, 8), n_lo=lo, n_hi=rng.randint(lo + 16, 150),
                    steps=rng.randint(200, 900), mix=rng.randint(1, 10 ** 6))
    boundary = rng.choice(["ldc", "periodic", "channel", "inflow"])
    l = _size(rng, 32, 420)
    m = _size(rng, 40, 200)
    n = max(40, min(200, int(m * rng.uniform(0.7, 1.4))))
    les = boundary in ("ldc", "periodic") and rng.random() < 0.2
    if boundary == "inflow":
        l = max(l, 2 * m)
    nu = {"ldc": 0.05, "periodic": 0.01, "channel": 0.1, "inflow": 0.02}[boundary]
    u0 = {"ldc": 0.1, "periodic": 0.05, "channel": 0.02, "inflow": 0.1}[boundary]
    obstacle = boundary == "inflow"
    cells = l * m * n
    if kind == "engine":
        storage, rounding, mixed = rng.choice([("f32", 0, 0)] * 3 + [("f64", 0, 0), ("f16", 1, 0), ("f16", 0, 0),
                                                                     ("bf16", 1, 0), ("f16", 0, 1), ("f32", 0, 2)])
        most = 4e11 / (38 * BYTES[storage] * cells)
        steps = int(min(2000, max(20, most * rng.uniform(0.3, 1.0))))
        return _engine(None, boundary, l, m, n, storage, steps, rounding=rounding, mixed=mixed, les=les,
                       wall_axis=rng.choice([2, 3]), obstacle=obstacle, nu=nu, u0=u0)
    prec = rng.choice(["sp", "sp", "dp"])
    if kind == "diag":
        return dict(kind="diag", boundary="inflow", l=max(l, 2 * m), m=m, n=n, prec=prec, steps=2 * rng.randint(2, 6),
                    les=False, obstacle=True, nu=0.02, u0=0.1)
    return _v1(None, boundary, l, m, n, prec, 2 * rng.randint(2, 20), les=les and boundary != "channel",
               obstacle=obstacle, nu=nu, u0=u0)


# ---- inputs -----------------------------------------------------------------


def _case(c, seed):
    r = random.Random(seed)
    nu, u0 = c["nu"] * r.uniform(0.9, 1.1), c["u0"] * r.uniform(0.9, 1.1)
    return Case(c["boundary"], c["l"], c["m"], c["n"], svisc=nu, u0=u0, init=1 if c["boundary"] == "periodic" else 0,
                obstacle=c["obstacle"], les=c["les"], wall_axis=c.get("wall_axis", 3))


def _inflow_u(seed):
    return 0.1 * random.Random(seed + 7).uniform(0.9, 1.1)


def _requests(c, seed):
    shape, r = random.Random(c["mix"]), random.Random(seed)
    out = []
    for q in range(c["count"]):
        n, half = shape.randint(c["n_lo"], c["n_hi"]), shape.random() < 0.5
        re = shape.uniform(100.0, 300.0) * r.uniform(0.9, 1.1)
        out.append(Request(n, re, "f16" if half else "f32", c["steps"], seed=seed % 65536 + q))
    return out


class _DeviceArray:
    """A device array of the simulation, for torch's view of it."""

    def __init__(self, buffer, shape, prec):
        self.buffer = buffer  # freed with its last reference: it has to outlive the view
        self.__cuda_array_interface__ = {"data": (buffer.ptr, False), "shape": shape, "strides": None, "version": 2,
                                         "typestr": "<f4" if prec == "sp" else "<f8"}


def _interior(buffer, shape, prec):
    view = torch.as_tensor(_DeviceArray(buffer, shape, prec), device="cuda")[1:-1, 1:-1, 1:-1]
    view.buffer = buffer
    return view


def _simulation(c, seed):
    case = _case(c, seed)
    if c["boundary"] == "inflow":
        case = case.with_(u_inflow=_inflow_u(seed))
    return Simulation(case, c["prec"], poison=False, device_init=True)


def prepare(case, seed):
    c = case
    if c["kind"] == "serve":
        return dict(kind="serve", requests=_requests(c, seed),
                    server=Server(4 << 30, policy="shortest", min_cells=4 << 20, chunk_ms=20.0))
    if c["kind"] == "engine":
        kw = dict(rounding=c["rounding"], mixed=c["mixed"], seed=seed % 65536)
        if c["boundary"] == "inflow":
            kw["u_inflow"] = _inflow_u(seed)
        eng = Engine(_case(c, seed), c["storage"], **kw)
        eng.step(c["before"])
        return dict(kind="engine", steps=c["steps"], engine=eng)
    sim = _simulation(c, seed)
    if c["kind"] == "diag":
        sim.step(c["steps"])
        sim.sync()
        return dict(kind="diag", sim=sim)
    views = {b.ptr: _interior(b, sim.case.shape, c["prec"]) for b in sim._a + sim._b}
    return dict(kind="v1", steps=c["steps"], sim=sim, views=views)


# ---- one pass -----------------------------------------------------------------


def run(state):
    if state["kind"] == "engine":
        eng = state["engine"]
        eng.step(state["steps"])
        return eng.fields()
    if state["kind"] == "v1":
        sim = state["sim"]
        sim.step(state["steps"])
        return [state["views"][p] for p in sim.pa]
    if state["kind"] == "diag":
        sim = state["sim"]
        u, w, v, den = sim.varm()
        c = sim.case
        return dict(diagno=sim.diagno(), varm=np.stack([u, w, v]), den=den, prof_i=sim.prof_i(), prof_j=sim.prof_j(),
                    prof_k=sim.prof_k(), probe=sim.probe(c.l // 2, c.m // 2, c.n // 2), draglift=sim.draglift())
    srv = state["server"]
    ids = [srv.submit(r) for r in state["requests"]]
    left = len(ids)
    while left:
        left -= len(srv.advance())
    diag = [srv.result(i)["diag"] for i in ids]
    for i in ids:
        srv.release(i)
    return diag


def work(case):
    """A step reads and writes every population of every cell once (38 values a cell); 250 operations a cell."""
    c = case
    if c["kind"] == "serve":
        rs = _requests(c, 1)
        return {"bytes": sum(38 * BYTES[r.storage] * r.cells * r.steps for r in rs),
                "flops": sum(250 * r.cells * r.steps for r in rs)}
    cells = c["l"] * c["m"] * c["n"]
    if c["kind"] == "engine":
        return {"bytes": 38 * BYTES[c["storage"]] * cells * c["steps"] + 32 * cells, "flops": 250 * cells * c["steps"]}
    s = 4 if c["prec"] == "sp" else 8
    if c["kind"] == "diag":
        return {"bytes": 19 * s * cells, "flops": 70 * cells}
    return {"bytes": 38 * s * cells * c["steps"], "flops": 250 * cells * c["steps"]}


# ---- the same flows in 64 bits, in plain torch ---------------------------------------

C = [(1, -1, 0), (1, 0, -1), (1, 1, 0), (1, 0, 1), (1, 0, 0), (0, 0, 1), (0, 1, 1), (0, 1, 0), (0, 1, -1),
     (-1, -1, 0), (-1, 0, -1), (-1, 1, 0), (-1, 0, 1), (-1, 0, 0), (0, 0, -1), (0, -1, -1), (0, -1, 0), (0, -1, 1),
     (0, 0, 0)]
OPP = [C.index((-x, -y, -z)) for x, y, z in C]
WGT = [{0: 1 / 3, 1: 1 / 18, 2: 1 / 36}[abs(x) + abs(y) + abs(z)] for x, y, z in C]


def _moments(f):
    drho = sum(f)
    inv = 1.0 / (1.0 + drho)
    u = [sum(s * g for s, g in ((C[d][a], f[d]) for d in range(19)) if s) * inv for a in range(3)]
    return drho, u


def _feq(drho, u, d):
    x, y, z = C[d]
    cu = x * u[0] + y * u[1] + z * u[2]
    return WGT[d] * (drho + (1.0 + drho) * (3.0 * cu + 4.5 * cu * cu - 1.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)))


def _edge(t, axis, side):
    """The outermost layer of t (k, j, i) along axis 0 x, 1 y, 2 z."""
    return t.select(2 - axis, 0 if side < 0 else t.shape[2 - axis] - 1)


class _Flow:
    """Shifted populations f - w of one flow in FP64, stepped with whole-array operations."""

    def __init__(self, boundary, l, m, n, nu, u0, init, les=False, wall_axis=3, u_in=0.1, solid=None, links=True):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.bc, self.les, self.links = boundary, les, links
        self.omega, self.lid = 2.0 / (6.0 * nu + 1.0), u0 / 6.0
        self.force = 4.0 * u0 * nu / (5.0 * m * m) if boundary == "channel" else 0.0
        self.walls = {"ldc": (0, 1, 2), "channel": (wall_axis - 1,)}.get(boundary, ())
        self.u_in = u_in
        self.solid = None if solid is None else torch.from_numpy(np.ascontiguousarray(solid)).to(dev)
        z = torch.zeros((n, m, l), dtype=torch.float64, device=dev)
        if init:
            # the reference's state: pi in single precision, the density's variation as a factor only
            pi = float(np.float32(math.pi))
            k, j, i = (2 * pi * (torch.arange(1, s + 1, dtype=torch.float64, device=dev) - 0.5) / s for s in (n, m, l))
            k, j, i = k[:, None, None], j[None, :, None], i[None, None, :]
            u = [u0 * torch.sin(i) * torch.cos(j) * torch.cos(k), -u0 * torch.cos(i) * torch.sin(j) * torch.cos(k), z]
            rho = 1.0 + u0 * u0 / 48.0 * (torch.cos(2 * i) + torch.cos(2 * j)) * (torch.cos(2 * k) + 2.0)
            self.f = [rho * _feq(z, u, d) for d in range(19)]
        else:
            self.f = [z.clone() for _ in range(19)]

    def _obstacle_in_place(self):
        """The reference's loop over the solid cells (k, j, i order): a_d(S) = a_opp(d)(S + c_d), except where
        S + c_d is itself solid and was visited before S."""
        s, old, new = self.solid, self.f, []
        for d in range(18):
            x, y, z = C[d]
            ahead = (-z, -y, -x)
            src, nb = torch.roll(old[OPP[d]], ahead, (0, 1, 2)), torch.roll(s, ahead, (0, 1, 2))
            earlier = z < 0 or (z == 0 and (y < 0 or (y == 0 and x < 0)))
            new.append(torch.where(s & ~nb if earlier else s, src, old[d]))
        self.f = new + [old[18]]

    def _pull(self):
        if self.bc == "inflow":
            last = [g[:, :, -1] for g in self.f]
            mom = [sum(C[d][a] * last[d] for d in range(18) if C[d][a]) for a in range(3)]
            inflow = [self.u_in, 0.0, 0.0]
        if self.solid is not None and not self.links:
            self._obstacle_in_place()
        out = []
        for d in range(19):
            x, y, z = C[d]
            p = torch.roll(self.f[d], (z, y, x), (0, 1, 2))
            own = self.f[OPP[d]]
            if self.bc == "inflow" and x:
                if x > 0:
                    p[:, :, 0] = _feq(0.0, inflow, d)
                else:
                    p[:, :, -1] = torch.roll(_feq(0.0, mom, d), (z, y), (0, 1))
            for a in self.walls:
                if C[d][a]:
                    _edge(p, a, -C[d][a]).copy_(_edge(own, a, -C[d][a]))
            if self.bc == "ldc" and d in (1, 10):  # the lid: pulls across the top wall
                _edge(p, 2, 1).add_(self.lid if d == 1 else -self.lid)
            if self.solid is not None and self.links and d < 18:
                p = torch.where(torch.roll(self.solid, (z, y, x), (0, 1, 2)), own, p)
            out.append(p)
        return out

    def step(self, steps):
        for _ in range(steps):
            f = self._pull()
            drho, u = _moments(f)
            w = self.omega
            if self.les:
                e = [_feq(drho, u, d) for d in range(18)]
                p = {}
                for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)):
                    p[a, b] = sum(C[d][a] * C[d][b] * (f[d] - e[d]) for d in range(18) if C[d][a] * C[d][b])
                q = sum((1.0 if a == b else 2.0) * v * v for (a, b), v in p.items()).sqrt()
                w = 1.0 / (0.5 / w + 0.5 * (18.0 * 0.1 ** 2 * q + (1.0 / w) ** 2).sqrt())
            self.f = [g + w * (_feq(drho, u, d) - g) for d, g in enumerate(f)]
            if self.force:
                for d in range(18):
                    if C[d][0]:
                        self.f[d] += C[d][0] * self.force * (1.0 + drho)

    def fields(self):
        drho, u = _moments(self.f)
        return [1.0 + drho] + u

    def diagno(self):
        rho, *u = self.fields()
        ke = 0.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
        return np.array([float(t.mean()) for t in (*u, rho, ke)])


def exact(case, seed):
    c = case
    if c["kind"] == "serve":
        out = []
        for r in _requests(c, seed):
            f = _Flow("ldc", r.n, r.n, r.n, r.svisc, r.u0, 0)
            f.step(r.steps)
            out.append(f.diagno())
        return out
    q = _case(c, seed)
    l, m, n = c["l"], c["m"], c["n"]
    solid = radius = centre = None
    if c["obstacle"]:
        obs, _, radius, centre = sphere_obstacle(l, m, n)
        solid = obs == 1
    u_in = _inflow_u(seed)
    f = _Flow(c["boundary"], l, m, n, q.svisc, q.u0, q.init, c["les"], c.get("wall_axis", 3), u_in, solid,
              links=c["kind"] == "engine")
    f.step(c["steps"] + c.get("before", 0))
    if c["kind"] == "engine":
        # a component that vanishes by symmetry has no value but the rounding's
        top = max(float(t.abs().max()) for t in f.fields()[1:])
        return [t.cpu().numpy() if float(t.abs().max()) > 1e-8 * top else None for t in f.fields()]
    if c["kind"] == "v1":
        return f.f
    rho, ux, uy, uz = (t.cpu().numpy() for t in f.fields())
    rows = np.stack([ux, uy, uz, rho], axis=-1)  # u, w (y velocity), v (z velocity), density
    j, k, i = m // 2, n // 2, l // 2
    force = np.zeros(3)
    near = torch.from_numpy(obs).to(f.f[0].device)
    for d in range(18):
        x, y, z = C[d]
        hit = torch.where((near == 0) & (torch.roll(near, (-z, -y, -x), (0, 1, 2)) == 1), f.f[d], torch.zeros_like(f.f[d]))
        force += 2.0 * np.array(C[d]) * float(hit.sum())
    return dict(diagno=f.diagno(), varm=np.stack([t.sum(axis=(1, 2)) / l for t in (ux, uy, uz)]),
                den=rho.sum(axis=(0, 2)) / l, prof_i=rows[k - 1, j - 1], prof_j=rows[k - 1, :, i - 1],
                prof_k=rows[:, j - 1, i - 1], probe=rows[k - 1, j - 1, i - 1], draglift=force / (u_in * u_in * radius))
