"""Handles that can have either rows (layout 0 where compact rows are faster
for one step and padded rows for two per launch): the same bits however the
calls cut the steps, and the rows that suit the calls."""
import numpy as np
import pytest

from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu

SIZES = {"f32": (70, 30, 24), "f64": (20, 12, 10), "mixed2": (40, 24, 24)}
CASES = {
    "ldc": dict(boundary="ldc"),
    "periodic": dict(boundary="periodic", init=1),
    "channel": dict(boundary="channel"),
    "channel-y": dict(boundary="channel", wall_axis=2),
    "inflow": dict(boundary="inflow"),
    "inflow-obstacle": dict(boundary="inflow", obstacle=True),
    "ldc-les": dict(boundary="ldc", les=True),
}


def make(form, kw, layout=0):
    l, m, n = SIZES[form]
    return Engine(Case(l=l, m=m, n=n, svisc=0.03, u0=0.1, **kw), "f64" if form == "f64" else "f32",
                  mixed=2 if form == "mixed2" else 0, layout=layout)


# (calls, compact rows after them): one step at a time; a long call; both in turn, odd and even between moves; twos
CALLS = [([1] * 20, True), ([1] * 20 + [6], False), ([4] + [1] * 17, True), ([1] * 17 + [7] + [1] * 18 + [9], False),
         ([1] * 16 + [2, 2], True), ([1] * 16 + [2] * 3 + [3], False)]


@pytest.mark.parametrize("form,name", [(f, c) for f in SIZES for c in CASES
                                       if (f, c) not in (("f64", "inflow-obstacle"), ("f64", "ldc-les"))])
def test_rows_follow_the_calls(gpu, form, name):
    """No obstacle fits the FP64 lattice, and FP64 LES takes one step per
    launch at these sizes."""
    print(f"[gpu] rows {form} {name}", flush=True)
    for calls, compact in CALLS:
        out = []
        with make(form, CASES[name]) as eng:
            assert eng.info()["nx"] % 16 == 0  # padded
            for c in calls:
                eng.step(c)
            assert (eng.info()["nx"] == eng.case.l + 2) == compact, calls
            out.append(eng.populations())
            rho, ux, _, _ = eng.fields()
        with make(form, CASES[name], layout=2) as eng:
            eng.step(sum(calls))
            out.append(eng.populations())
            ref = eng.fields()
        assert np.isfinite(out[0]).all() and np.any(out[0] != 0)
        assert np.array_equal(out[0], out[1]), calls
        assert np.array_equal(rho, ref[0]) and np.array_equal(ux, ref[1])


def test_state_set_and_restored_across_moves(gpu, tmp_path):
    """Files and populations written in one kind of rows and read in the other."""
    kw = CASES["inflow-obstacle"]
    with make("f32", kw) as a, make("f32", kw) as b:
        a.step(8)
        a.save_raw(tmp_path / "padded.bin", 8)
        for _ in range(20):
            a.step(1)
        assert a.info()["nx"] == a.case.l + 2
        a.save_raw(tmp_path / "compact.bin", 28)
        a.step(3)
        b.restore_raw(tmp_path / "padded.bin")
        for _ in range(20):
            b.step(1)
        assert b.info()["nx"] == b.case.l + 2
        b.restore_raw(tmp_path / "compact.bin")
        b.step(3)
        assert np.array_equal(a.populations(), b.populations())
        new = [np.random.default_rng(d).uniform(-0.01, 0.01, (24, 30, 70)) for d in range(19)]
        for eng, calls in ((a, [6]), (b, [1] * 6)):
            for d in range(19):
                eng.set_population(d, new[d])
            for c in calls:
                eng.step(c)
        assert np.array_equal(a.populations(), b.populations())
