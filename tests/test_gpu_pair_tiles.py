"""collide_pair with tiles of given rows and planes against one step per launch:
every boundary, force, obstacle, LES and storage form, tiles of one row up to
the most, several planes a block with a short last range, and the last rows and
cells in tiles of their own.  The library's choice for lattices of this size
would be tiles of a row and a plane, or one step per launch."""
import numpy as np
import pytest

from bgk3d_gpu_amd import runtime as rt
from bgk3d_gpu_amd import serving as S
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu

STORAGE = {"f32": ("f32", 0, 13), "f64": ("f64", 0, 8), "mixed2": ("f32", 2, 9)}  # most rows of a tile
FORMS = {
    "ldc": dict(boundary="ldc"),
    "periodic": dict(boundary="periodic"),
    "walls-y-force-x": dict(boundary="channel", wall_axis=2),
    "walls-y-force-z": dict(boundary="channel", wall_axis=2, force_axis=3),
    "walls-z-force-x": dict(boundary="channel"),
    "walls-z-force-y": dict(boundary="channel", force_axis=2),
    "walls-z-force-z": dict(boundary="channel", force_axis=3),
    "inflow": dict(boundary="inflow"),
    "inflow-obstacle": dict(boundary="inflow", obstacle=True),
    "periodic-obstacle": dict(boundary="periodic", obstacle=True),
}


def tilings(most):
    """(l, m, n), rows, planes: full and narrow columns, narrow only, two full
    ones (the second short), one cell in a narrow one; one row or plane over."""
    return [((70, most + 1, 9), most, 4), ((20, 2 * most + 1, 7), most - 1, 3), ((100, 5, 9), 2, 2),
            ((64, 2 * most, 8), most, 8), ((129, 3, 6), 1, 5)]


def run(case, storage, mixed, calls, launch, **kw):
    rng = np.random.default_rng(case.l)
    shape = (case.n, case.m, case.l)
    with Engine(case, storage, layout=1, mixed=mixed, **kw) as eng:
        eng.set_launch(*launch)
        info = eng.launch_info()
        assert info["steps_per_launch"] == launch[0]
        if launch[0] == 2:
            assert (info["tile_rows"], info["tile_planes"]) == launch[1:]
        for d in range(19):
            eng.set_population(d, rng.uniform(-0.004, 0.004, shape))
        for c in calls:
            eng.step(c)
        return eng.populations()


@pytest.mark.parametrize("les", [False, True], ids=["", "les"])
@pytest.mark.parametrize("storage", list(STORAGE))
@pytest.mark.parametrize("form", list(FORMS))
def test_tiles_match_single_steps(gpu, form, storage, les):
    st, mixed, most = STORAGE[storage]
    for (l, m, n), rows, planes in tilings(most):
        kw = {}
        if "obstacle" in form:
            m, n, kw = max(m, 14), max(n, 14), dict(radius=2)
        print(f"[gpu] tiles {form} {storage} les={les} {l}x{m}x{n} rows {rows} planes {planes}", flush=True)
        case = Case(l=l, m=m, n=n, svisc=0.03, u0=0.1, les=les, **FORMS[form])
        two = run(case, st, mixed, (7,), (2, rows, planes), **kw)
        one = run(case, st, mixed, (7,), (1,), **kw)
        assert np.isfinite(one).all() and np.ptp(one[18]) > 0
        assert np.array_equal(two, one)


def test_launch_can_be_given_back(gpu):
    """0 restores the choice; forms that cannot take two steps per launch, and
    tiles that no block holds, are refused."""
    case = Case("ldc", 70, 30, 24, svisc=0.03, u0=0.1)
    with Engine(case, "f32") as eng, Engine(case, "f32") as ref:
        first = eng.launch_info()
        assert first["steps_per_launch"] == 2 and not first["compact"]
        for launch in ((1,), (2, 3, 5), (0,), (1,), (0,)):
            eng.set_launch(*launch)
            assert eng.launch_info()["compact"] == (launch[0] == 1) or launch == (0,)
            eng.step(6)
        assert eng.launch_info() == first
        ref.step(30)
        assert np.array_equal(eng.populations(), ref.populations())
        for bad in ((2, 14, 1), (2, 1, 25), (1, 3, 0), (0, 0, 2), (3,), (-1,)):
            with pytest.raises(rt.BGKError):
                eng.set_launch(*bad)
        assert eng.launch_info() == first
    for storage, layout in (("f16", 1), ("bf16", 0), ("f32", 2)):
        with Engine(case, storage, layout=layout) as eng:
            with pytest.raises(rt.BGKError):
                eng.set_launch(2)
            eng.step(2)
            assert eng.launch_info()["steps_per_launch"] == 1


@pytest.mark.parametrize("steps", [10, 11])
def test_pairs_of_several_requests(gpu, steps):
    """Requests of one two-step launch: tiles for their share of the GPU."""
    reqs = [S.Request(n, 150.0 + n, st, steps, keep=True) for st, ns in (("f32", (24, 64, 31, 85, 35)),
                                                                         ("f64", (20, 30, 61, 26))) for n in ns]
    with S.Server(2 << 30, 50) as srv:
        ids = [srv.submit(r) for r in reqs]
        assert sorted(srv.advance()) == sorted(ids)
        assert srv.stats()["launches"] == 2 * ((steps + 1) // 2)
        for rid, r in zip(ids, reqs):
            with Engine(r.case(), r.storage, layout=1) as eng:
                eng.set_launch(1)
                eng.step(steps)
                assert np.array_equal(srv.populations(rid, r.n), eng.populations()), (r.n, r.storage)


@pytest.mark.parametrize("name", ["ldc", "periodic", "inflow", "ldc-les"])
@pytest.mark.parametrize("size,storage", [((64, 60, 60), "f32"), ((80, 80, 80), "f32"), ((75, 75, 75), "f64")],
                         ids=["stream-f32", "plain-f32", "plain-f64"])
def test_plain_and_streaming_stores(gpu, size, storage, name):
    """Lattices below 80 MB (streaming stores) and just above (plain ones), two
    steps per launch throughout."""
    case = Case(name.split("-")[0], *size, svisc=0.02, u0=0.1, init=1 if name == "periodic" else 0, les="les" in name)
    out = []
    for launch in (2, 1):
        with Engine(case, storage, layout=1) as eng:
            eng.set_launch(launch)
            assert eng.launch_info()["steps_per_launch"] == launch
            assert (eng.info()["bytes"] >= 80000000) == (size[0] != 64)
            eng.step(6)
            out.append([eng.population(d) for d in (0, 5, 10, 18)])
    assert np.any(out[0][0] != 0) and np.array_equal(out[0], out[1])
