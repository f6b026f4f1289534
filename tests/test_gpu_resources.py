"""What calls share and keep: the staging of bgk_fields, the scratch of the
diagnostics, device memory."""
import ctypes
import threading

import numpy as np
import pytest

from bgk3d_gpu_amd import engine as E
from bgk3d_gpu_amd import runtime as rt
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine
from bgk3d_gpu_amd.simulation import Simulation
from test_gpu_v1_parity import per_cell_moments

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so").hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_fields_from_several_threads(gpu):
    """One handle's fields asked for by four threads at once, each for another
    set of them (so that the staging grows while others wait for it)."""
    case = Case("periodic", 96, 80, 70, svisc=0.02, u0=0.05, init=1)
    with Engine(case, "f32") as eng:
        eng.step(4)
        want = eng.fields()
    with Engine(case, "f32") as eng:
        eng.step(4)
        wrong = []

        def ask(which):
            for _ in range(20):
                got = [np.empty((case.n, case.m, case.l)) if q in which else None for q in range(4)]
                rc = eng.L.bgk_fields(eng.h, *[None if g is None else g.ctypes.data for g in got])
                if rc or not all(np.array_equal(got[q], want[q]) for q in which):
                    wrong.append((which, rc))

        threads = [threading.Thread(target=ask, args=(w,)) for w in ((0,), (1, 3), (0, 1, 2, 3), (2, 3, 0))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong, (wrong[:4], E.lib().bgk_last_error())


def test_fields_after_a_refused_handle(gpu):
    """A lattice that cannot be allocated (19 TB) leaves the other handles of
    the thread as they were."""
    with Engine(Case("ldc", 20, 20, 20, svisc=0.05, u0=0.1), "f32") as eng:
        eng.step(2)
        want = eng.fields()
        with pytest.raises(rt.BGKError):
            Engine(Case("ldc", 4000, 4000, 4000, svisc=0.05, u0=0.1), "f64")
        assert np.array_equal(eng.fields(), want)


def test_varm_keeps_little_device_memory(gpu):
    """Six million rows: their sums would take 192 MB that stay until the
    process ends; the scratch is 8 MB."""
    sim = Simulation(Case("periodic", 1, 3000, 2000), "sp", poison=False, device_init=True)
    try:
        sim.diagno()
        before = free_bytes()
        sim.varm()
        assert before - free_bytes() <= 16 << 20
    finally:
        sim.close()


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("size", [(2, 700, 400), (1, 262144, 2), (2, 511, 514)], ids=lambda s: "x".join(map(str, s)))
def test_varm_in_several_passes(gpu, size, prec):
    """More rows than the scratch holds at a time: two passes, the second one
    short; one plane a pass; one plane left over."""
    case = Case("periodic", *size)
    print(f"[gpu] varm in passes {prec} {size}", flush=True)
    rng = np.random.default_rng(sum(size))
    sim = Simulation(case, prec, poison=False, device_init=True)
    try:
        G = rng.uniform(-0.01, 0.01, (19,) + case.shape).astype(sim.R)
        sim.set_state(G)
        u, w, v, den = sim.varm()
    finally:
        sim.close()
    per = {q: a.astype(np.float64) for q, a in per_cell_moments(G, case, prec).items()}
    rvol = float(np.float32(1.0) / np.float32(case.l))
    # FP64 sums of at most 524,288 terms, by a wave and a block at a time: 1e-12 of the sum of magnitudes is
    # more than 10 times the rounding of the longest chain of additions (2048 of them, and a tree)
    for got, q in ((u, "u"), (w, "w"), (v, "v")):
        mag = np.abs(per[q]).sum(axis=(1, 2)) * rvol
        assert np.all(np.abs(got - per[q].sum(axis=(1, 2)) * rvol) <= 1e-12 * mag), q
    np.testing.assert_allclose(den, per["rho"].sum(axis=(0, 2)) * rvol, rtol=1e-12)


def test_calls_after_a_refused_handle(gpu):
    """Stepping, creating, serving and moving rows after one."""
    from bgk3d_gpu_amd import serving as S

    case = Case("periodic", 70, 30, 24, svisc=0.03, u0=0.1, init=1)

    def refuse():
        with pytest.raises(rt.BGKError):
            Engine(Case("ldc", 4000, 4000, 4000, svisc=0.05, u0=0.1), "f64")

    with Engine(case, "f32") as eng:
        refuse()
        eng.step(2)
        refuse()
        eng.time_steps(4)
        refuse()
        eng.set_launch(1)
        refuse()
        with Engine(case, "f32") as other:
            other.step(6)
            assert np.array_equal(eng.populations(), other.populations())
        with S.Server(1 << 28, 10) as srv:
            rid = srv.submit(S.Request(30, 200.0, "f32", 10))
            refuse()
            assert srv.advance() == [rid]
