"""diagno on rows that a block takes (few of them) and on rows that a wave
takes: row counts and lengths on either side of the lines between them."""
import numpy as np
import pytest

from bgk3d_gpu_amd import runtime as rt
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine
from bgk3d_gpu_amd.simulation import Simulation
from test_gpu_reductions import test_reductions_on_edge_sizes as reductions

pytestmark = pytest.mark.gpu

SIZES = [(64, 16, 16), (65, 1, 1), (255, 3, 2), (256, 16, 16), (257, 16, 16), (129, 257, 1), (512, 1, 257),
         (513, 32, 16), (513, 27, 19), (2000, 3, 5)]


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_long_rows(gpu, size, prec):
    reductions(gpu, size, prec)


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_every_entry_gives_the_same_means(gpu, size):
    """diagno_gpu, diagno_gpu_noalloc and the handle's diagno: the same sums in
    the same order."""
    case = Case("periodic", *size, svisc=0.02, u0=0.05, init=1)
    sim = Simulation(case, "dp", poison=False, device_init=True)
    try:
        want, got = sim.diagno(), np.zeros(5)
        rt.check(sim.lib.diagno_gpu_noalloc(sim.pa, case.l, case.m, case.n, sim.nx, sim.ny, sim.Rc(sim.cte1),
                                            got.ctypes.data), "diagno_gpu_noalloc")
    finally:
        sim.close()
    with Engine(case, "f64") as eng:
        assert np.array_equal(eng.diagno(), want)
    assert np.array_equal(got, want)
