"""bgk_plan: the rows and the memory a handle takes (no GPU needed)."""
import pytest

from bgk3d_gpu_amd import runtime as rt
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import plan


CHOICE = [((130, 130, 130), "f32"), ((130, 130, 130), "f64"), ((420, 199, 180), "f32"), ((97, 97, 140), "f32"),
          ((97, 97, 140), "f64"), ((1000, 1000, 1000), "f32"), ((1000, 1000, 1000), "f64")]


@pytest.mark.parametrize("size,storage", CHOICE, ids=lambda s: s if isinstance(s, str) else "x".join(map(str, s)))
def test_padded_rows_leave_room(size, storage):
    """Lattices whose padded rows take more memory than the compact ones that
    suit one step: these are chosen where the room left is short of eight times
    the difference and 64 MB."""
    case = Case("periodic", *size, svisc=0.02, u0=0.05, init=1)
    compact = plan(case, storage, layout=2)["bytes"]
    padded = plan(case, storage, layout=1)["bytes"]
    extra, cells = padded - compact, case.cells
    assert extra > 0
    edge = padded + 8 * extra + (64 << 20)
    for free in (0, compact, padded, padded + extra, edge - 1, edge, 2 * edge, 1 << 60):
        p = plan(case, storage, free)
        assert p["bytes"] == (padded if free >= edge else compact)
        assert p["steps_per_launch"] == 2 - p["compact"] == (2 if free >= edge else 1)
        if free >= compact:
            assert 9 * (free - p["bytes"]) >= 8 * (free - compact)
        if free >= padded and not p["compact"]:
            # the calls of a handle that had the room for them beside compact rows
            assert free - p["bytes"] >= min(8 * cells, free - compact)


def test_rows_without_a_choice_do_not_look_at_the_room():
    case = Case("ldc", 64, 64, 64)
    assert plan(case, "f32", 0) == plan(case, "f32")          # padded rows are right for one step too
    assert plan(case, "f32", 0, layout=1) == plan(case, "f32", layout=1)
    assert plan(Case("ldc", 130, 130, 130), "f32", 0, layout=1)["steps_per_launch"] == 2
    assert plan(Case("ldc", 130, 130, 130), "f16", 0)["steps_per_launch"] == 1


def test_plan_rejects_what_create_rejects():
    for case, kw in ((Case("channel", 8, 8, 8, wall_axis=1), {}), (Case("ldc", 8, 8, 8), dict(layout=3)),
                     (Case("ldc", 8, 8, 8), dict(obstacle=1)), (Case("ldc", 8, 8, 8), dict(mixed=1))):
        with pytest.raises(rt.BGKError):
            plan(case, **kw)
