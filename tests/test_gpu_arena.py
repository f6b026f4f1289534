"""The server's arena and launches: what a request holds beyond request_bytes,
and the holes that finished ones leave, keep nobody waiting; requests of one
step per launch share launches up to 512 MB."""
import numpy as np
import pytest

from bgk3d_gpu_amd import serving as S
from bgk3d_gpu_amd.engine import Engine

pytestmark = pytest.mark.gpu


def finish(srv, rid, most=200):
    for _ in range(most):
        if srv.status(rid)[0] == "done":
            return
        srv.advance()
    pytest.fail(f"request {rid} is still {srv.status(rid)}")


def alone(r, dirs):
    with Engine(r.case(), r.storage, rounding=0) as eng:
        eng.step(r.steps)
        return [eng.population(d) for d in dirs]


@pytest.mark.parametrize("n,storage", [(87, "f32"), (75, "f64")])
@pytest.mark.parametrize("steps", [20, 21, 22, 23])
def test_kept_request_leaves_room(gpu, n, storage, steps):
    """A kept request took the room of two steps per launch while it was
    alone; the next one fits beside its request_bytes.  Both lattices' turns,
    direction 19's among them."""
    reqs = [S.Request(n, 200.0, storage, steps, keep=True), S.Request(n, 300.0, storage, 9, keep=True)]
    need = [S.request_bytes(r) for r in reqs]
    print(f"[gpu] arena: kept {storage} {n} {steps} steps", flush=True)
    with S.Server(sum(need), 50) as srv:
        ids = [srv.submit(reqs[0])]
        finish(srv, ids[0])
        assert srv.stats()["bytes_used"] > need[0]
        ids.append(srv.submit(reqs[1]))
        finish(srv, ids[1])
        assert srv.stats()["bytes_used"] == sum(need)
        for rid, r in zip(ids, reqs):
            dirs = (0, 5, 10, 18)
            for d, ref in zip(dirs, alone(r, dirs)):
                assert np.array_equal(srv.population(rid, d, n), ref), (rid, d)


@pytest.mark.parametrize("policy", ["all", "shortest"])
def test_later_request_joins_at_once(gpu, policy):
    """A request that comes while another runs with more than its
    request_bytes is admitted in the same chunk, and neither's result changes."""
    reqs = [S.Request(87, 200.0, "f32", 45, keep=True), S.Request(87, 300.0, "f32", 31, keep=True)]
    with S.Server(sum(S.request_bytes(r) for r in reqs), 10, policy=policy, min_cells=1 << 30) as srv:
        ids = [srv.submit(reqs[0])]
        srv.advance()
        ids.append(srv.submit(reqs[1]))
        srv.advance()
        assert srv.status(ids[1]) == ("active", 10)
        for rid in ids:
            finish(srv, rid)
        for rid, r in zip(ids, reqs):
            dirs = (1, 7, 14, 18)
            for d, ref in zip(dirs, alone(r, dirs)):
                assert np.array_equal(srv.population(rid, d, r.n), ref), (rid, d)


def test_holes_are_gathered(gpu):
    """Four lattices side by side, the first and the third released: a fifth
    that fits neither hole, but both, is admitted, and the two that stay keep
    their populations (FP16 and FP32, moved by less and by more than their own
    size)."""
    sizes = [(60, "f16", 12), (100, "f32", 7), (90, "f16", 15), (50, "f32", 8)]
    reqs = [S.Request(n, 200.0, st, steps, rounding=0, keep=True) for n, st, steps in sizes]
    need = [S.request_bytes(r) for r in reqs]
    last = S.Request(max(n for n in range(60, 100) if S.request_bytes(S.Request(n, 200.0, "f16")) <= need[0] + need[2]),
                     200.0, "f16", 5, rounding=0, keep=True)
    assert S.request_bytes(last) > max(need[0], need[2])
    with S.Server(sum(need), 50) as srv:
        ids = [srv.submit(r) for r in reqs]
        for rid in ids:
            finish(srv, rid)
        srv.release(ids[0])
        srv.release(ids[2])
        rid = srv.submit(last)
        finish(srv, rid)
        for q, r in ((ids[1], reqs[1]), (ids[3], reqs[3]), (rid, last)):
            dirs = (0, 6, 13, 18)
            for d, ref in zip(dirs, alone(r, dirs)):
                assert np.array_equal(srv.population(q, d, r.n), ref), (r.n, d)


def test_one_step_requests_share_launches(gpu):
    """Two FP16 requests of 436 MB together, more than the last-level cache
    holds: one launch a step, which fills the GPU."""
    reqs = [S.Request(140, 200.0 + q, "f16", 10) for q in range(2)]
    assert 1 << 28 < sum(S.request_bytes(r) for r in reqs) < 1 << 29
    with S.Server(1 << 30, 10) as srv:
        for r in reqs:
            srv.submit(r)
        assert len(srv.advance()) == 2
        assert srv.stats()["launches"] == 10


def test_a_released_request_claims_nothing(gpu):
    """The rows of two steps per launch are taken while every queued request
    fits beside them: one that was released from the queue, or that ended,
    counts no longer."""
    r, big = S.Request(87, 200.0, "f32", 6), S.Request(120, 200.0, "f32", 6)
    need = S.request_bytes(r)
    with S.Server(need + S.request_bytes(big), 3) as srv:
        for turn in range(3):
            a, b = srv.submit(r), srv.submit(big)
            if turn:
                srv.release(b)
            srv.advance()
            used = srv.stats()["bytes_used"]
            assert used > need if turn else used == need + S.request_bytes(big), turn
            finish(srv, a)
            if not turn:
                finish(srv, b)
            assert srv.stats()["bytes_used"] == 0
            for rid in (a, b)[:1 if turn else 2]:
                srv.release(rid)
