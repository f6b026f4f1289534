"""diagno and varm of the reference-compatible ABI at the edges of their row
mapping (a wave per row of cells, four to a block): rows of one cell, one wave
and one more, row counts that fill no block, exactly one, or more than the
1024 blocks of diagno hold one row each.
"""
import numpy as np
import pytest

from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.simulation import Simulation
from test_gpu_v1_parity import per_cell_moments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("size", [(1, 1, 1), (63, 1, 3), (64, 2, 2), (65, 5, 1), (130, 3, 7), (5, 300, 17)],
                         ids=lambda s: "x".join(map(str, s)))
def test_reductions_on_edge_sizes(gpu, size, prec):
    case = Case("periodic", *size)
    print(f"[gpu] reductions {prec} {size}", flush=True)
    rng = np.random.default_rng(sum(size))
    sim = Simulation(case, prec)
    try:
        G = rng.uniform(-0.01, 0.01, (19,) + case.shape).astype(sim.R)
        sim.set_state(G)
        dg = sim.diagno()
        u, w, v, den = sim.varm()
    finally:
        sim.close()
    per = {q: a.astype(np.float64) for q, a in per_cell_moments(G, case, prec).items()}
    rvol = float(np.float32(1.0) / np.float32(case.l))
    # FP64 sums of at most 25,500 terms: 1e-12 of the sum of magnitudes is 40 times their worst rounding
    for got, q in ((u, "u"), (w, "w"), (v, "v")):
        mag = np.abs(per[q]).sum(axis=(1, 2)) * rvol
        assert np.all(np.abs(got - per[q].sum(axis=(1, 2)) * rvol) <= 1e-12 * mag), q
    np.testing.assert_allclose(den, per["rho"].sum(axis=(0, 2)) * rvol, rtol=1e-12)
    for got, q in zip(dg, ("u", "w", "v", "rho")):
        assert abs(got - per[q].mean()) <= 1e-12 * np.abs(per[q]).mean(), q
