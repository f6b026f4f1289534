"""Two steps per launch (handle API, collide_pair): the same bits as the oracle
and as single steps, at the edges of its tiles.

Tiles are 64 cells in x and up to 13 rows (8 or 9 with FP64 arithmetic), cut
into ranges of planes; the sizes below leave one cell, one row or one plane
over, fit exactly, or are smaller than a tile's border.
"""
import numpy as np
import pytest

import oracle_support as O
from bgk3d_gpu_amd import serving as S
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 2, 2), (63, 1, 2), (64, 13, 3), (65, 14, 1), (66, 27, 5), (128, 8, 9), (129, 9, 4)]
CASES = {
    "ldc": dict(boundary="ldc", svisc=0.05, u0=0.1),
    "periodic": dict(boundary="periodic", svisc=0.02, u0=0.05, init=1),
    "channel": dict(boundary="channel", svisc=0.1, u0=0.5),
    "inflow": dict(boundary="inflow", svisc=0.05, u0=0.1),
    "ldc_les": dict(boundary="ldc", svisc=0.01, u0=0.1, les=True),
}


@pytest.mark.parametrize("storage", ["f32", "f64"])
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_pairs_match_oracle(gpu, size, name, storage):
    """Six steps in one call (three launches) and in calls of 1, 2 and 3."""
    case = Case(l=size[0], m=size[1], n=size[2], **CASES[name])
    print(f"[gpu] pairs {name} {storage} {size}", flush=True)
    out = []
    for chunks in ((6,), (1, 2, 3)):
        with Engine(case, storage, layout=1) as eng:
            for c in chunks:
                eng.step(c)
            out.append(eng.populations())
    prec = "sp" if storage == "f32" else "dp"
    A = O.new_lattice(case.l, case.m, case.n, prec)
    B = O.new_lattice(case.l, case.m, case.n, prec)
    O.init(A, case.l, case.m, case.n, prec, mode=case.init, u00=case.u00)
    O.run(case.boundary, A, B, case.l, case.m, case.n, 6, prec=prec, svisc=case.svisc, u0=case.u0, les=case.les,
          cte_s=case.cte_s)
    ref = A[:, 1:-1, 1:-1, 1:-1].astype(np.float64)
    assert np.array_equal(out[0], ref), f"max |diff| {np.abs(out[0] - ref).max()}"
    assert np.array_equal(out[1], ref)


@pytest.mark.parametrize("storage,mixed", [("f32", 0), ("f64", 0), ("f32", 2)])
@pytest.mark.parametrize("kw", [dict(boundary="periodic", init=1, obstacle=True), dict(boundary="inflow", obstacle=True),
                                dict(boundary="channel", wall_axis=2), dict(boundary="channel", wall_axis=2, force_axis=3),
                                dict(boundary="channel", force_axis=2), dict(boundary="ldc")],
                         ids=["periodic-obstacle", "inflow-obstacle", "walls-y", "walls-y-force-z", "force-y", "ldc"])
def test_pairs_match_single_steps(gpu, kw, storage, mixed):
    """Forms the oracle's runs above leave out, against step(1) calls: links of
    an obstacle that spans several tiles, walls in y with z periodic, MIXED2."""
    case = Case(l=70, m=30, n=24, svisc=0.03, u0=0.1, **kw)
    print(f"[gpu] pairs against singles {kw} {storage} mixed={mixed}", flush=True)
    out = []
    for chunks in ((20,), (1,) * 20):
        with Engine(case, storage, layout=1, mixed=mixed) as eng:
            for c in chunks:
                eng.step(c)
            out.append(eng.populations())
    assert np.isfinite(out[0]).all() and np.any(out[0] != 0)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("storage,mixed", [("f32", 0), ("f64", 0), ("f32", 2)])
@pytest.mark.parametrize("name", ["ldc", "periodic", "channel", "inflow"])
@pytest.mark.parametrize("size", [(32, 27, 3), (31, 1, 2), (33, 3, 4), (96, 53, 3), (95, 17, 5), (160, 19, 2)],
                         ids=lambda s: "x".join(map(str, s)))
def test_narrow_tiles_match_single_steps(gpu, size, name, storage, mixed):
    """The tiles of 32 cells and two rows per wave that take a row's last 1 ... 32
    cells: none but them, beside one or two of 64, one cell too many for them;
    rows that end in the first or the second half of a wave, in a tile of
    their own, or in a full tile."""
    case = Case(l=size[0], m=size[1], n=size[2], **CASES[name])
    print(f"[gpu] narrow tiles {name} {storage} mixed={mixed} {size}", flush=True)
    out = []
    for chunks in ((6,), (1,) * 6):
        with Engine(case, storage, layout=1, mixed=mixed) as eng:
            for c in chunks:
                eng.step(c)
            out.append(eng.populations())
    assert np.isfinite(out[0]).all() and np.any(out[0] != 0)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("storage,mixed", [("f64", 0), ("f32", 2)])
@pytest.mark.parametrize("kw", [dict(boundary="ldc"), dict(boundary="periodic", init=1),
                                dict(boundary="inflow", obstacle=True)], ids=["ldc", "periodic", "inflow-obstacle"])
def test_les_in_fp64_matches_single_steps(gpu, kw, storage, mixed):
    """LES with FP64 arithmetic, in full and in narrow tiles."""
    case = Case(l=70, m=30, n=24, svisc=0.01, u0=0.1, les=True, **kw)
    print(f"[gpu] LES pairs {kw} {storage} mixed={mixed}", flush=True)
    out = []
    for chunks in ((8,), (1,) * 8):
        with Engine(case, storage, layout=1, mixed=mixed) as eng:
            for c in chunks:
                eng.step(c)
            out.append(eng.populations())
    assert np.isfinite(out[0]).all() and np.any(out[0] != 0)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("n,storage", [(87, "f32"), (75, "f64")])
def test_server_takes_the_layout_that_fits(gpu, n, storage):
    """A served request whose two-step layout needs more bytes than
    request_bytes: admitted into exactly that much with one step per launch,
    into more with two, with the same populations."""
    out = []
    need = S.request_bytes(S.Request(n, 200.0, storage, 30))
    for budget in (need, 3 * need):
        srv = S.Server(budget, chunk_steps=7)
        try:
            rid = srv.submit(S.Request(n, 200.0, storage, 30, keep=True))
            while rid not in srv.advance():
                pass
            out.append([srv.population(rid, d, n) for d in (0, 5, 18)])
        finally:
            srv.close()
    assert np.isfinite(out[0]).all() and np.any(out[0][0] != 0)
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("size,storage", [((64, 60, 60), "f32"), ((80, 80, 80), "f32"), ((112, 112, 112), "f32"),
                                          ((90, 90, 90), "f64")], ids=["stream", "low", "high", "f64"])
@pytest.mark.parametrize("name", ["ldc", "periodic", "inflow"])
def test_stores_that_stay_in_cache(gpu, size, storage, name):
    """Plain stores where both lattices fit the last-level cache (80 ... 256 MB),
    against single steps, which always stream."""
    case = Case(l=size[0], m=size[1], n=size[2], **CASES[name])
    print(f"[gpu] cached stores {name} {storage} {size}", flush=True)
    out = []
    for chunks in ((4,), (1,) * 4):
        with Engine(case, storage, layout=1) as eng:
            for c in chunks:
                eng.step(c)
            out.append([eng.population(d) for d in (0, 5, 10, 18)])
    assert np.isfinite(out[0]).all() and np.any(out[0][0] != 0)
    assert np.array_equal(out[0], out[1])
