"""What calls share and keep: the staging of bgk_fields, the scratch of the
diagnostics, device memory."""
import threading

import numpy as np
import pytest

from bgk3d_gpu_amd import engine as E
from bgk3d_gpu_amd import runtime as rt
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu


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
    """A lattice that cannot be allocated (17 TB) leaves the other handles of
    the thread as they were."""
    with Engine(Case("ldc", 20, 20, 20, svisc=0.05, u0=0.1), "f32") as eng:
        eng.step(2)
        want = eng.fields()
        with pytest.raises(rt.BGKError):
            Engine(Case("ldc", 4000, 4000, 4000, svisc=0.05, u0=0.1), "f64")
        assert np.array_equal(eng.fields(), want)
