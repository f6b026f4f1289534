"""bench.py reports the steps per launch and the rows that the handle has."""
import pytest

import bench
from bgk3d_gpu_amd.cases import Case
from bgk3d_gpu_amd.engine import plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,storage,mixed,want", [
    ((64, 64, 64), "f32", 2, (1, False)),     # padded rows, one step per launch
    ((126, 64, 64), "f32", 0, (2, False)),    # two steps per launch on padded rows of l + 2 cells
    ((99, 80, 60), "f32", 0, (1, True)),      # compact rows
    ((130, 130, 130), "f32", 0, (2, False)),
    ((64, 64, 64), "f16", 0, (1, False)),
], ids=["padded-one", "padded-no-wider", "compact", "pair", "f16"])
def test_steps_per_launch_of_a_run(gpu, size, storage, mixed, want):
    case = Case("periodic", *size, svisc=0.02, u0=0.05, init=1)
    _, _, _, info = bench.bench_engine(case, storage, 6, 2, mixed=mixed)
    assert (info["steps_per_launch"], info["compact"]) == want
    assert (info["nx"] == size[0] + 2) == (want[1] or size[0] == 126)
    p = plan(case, storage, mixed=mixed)
    assert (p["steps_per_launch"], p["compact"]) == want and p["bytes"] == info["bytes"]
    if want[0] == 2:  # a single step has a launch of its own
        assert bench.bench_engine(case, storage, 1, 2, mixed=mixed)[3]["steps_per_launch"] == 1
