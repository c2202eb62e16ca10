"""The request loop with preconditioned requests: its settings are those of its creation."""
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1
SHAPES = [((64, 50, 48), 0), ((48, 50, 64), 4), ((40, 30, 30), 2)]


def solo_and_requests():
    masks = [F.generate_ellipsoids(s, 12.0, 0.35, 0.6, 4 + i) for i, (s, _) in enumerate(SHAPES)]
    ps = [T.make_params(d, CG, "mixed", 1e-9, 20000) for _, d in SHAPES]
    c = T.Context(0)
    try:
        solo = [c.volume(m).solve(p)[0] for m, p in zip(masks, ps)]
    finally:
        c.close()
    return solo, masks, ps


def serve(s, masks, ps):
    tickets = [s.submit(m, p) for m, p in zip(masks, ps)]
    got = {}
    for _ in tickets:
        t, r, _ = s.wait(60000)
        got[t] = r
    return [got[t] for t in tickets]


@pytest.mark.parametrize("at_start,later", [("2", "0"), ("0", "2"), ("2", "1")])
def test_form_of_the_passes_is_that_of_the_servers_creation(monkeypatch, at_start, later):
    """The preconditioner's levels lie in the Y vector where the passes do not use it, so a change of
    FAST_TAU_RB_STAGED while a server lives must not bring that vector into use: every result is
    the solo solve's, bit for bit."""
    solo, masks, ps = solo_and_requests()
    monkeypatch.setenv("FAST_TAU_RB_STAGED", at_start)
    c = T.Context(0)
    s = T.Server(c, hbm_budget=256 << 20)
    try:
        monkeypatch.setenv("FAST_TAU_RB_STAGED", later)
        for r, q in zip(serve(s, masks, ps), solo):
            assert r.status == 0 and (r.tau, r.iterations) == (q.tau, q.iterations)
    finally:
        s.close()
        c.close()


def test_server_within_the_budget_of_the_jacobi_form(monkeypatch):
    """With separate Y and Q passes the levels need a plane of their own (8 bytes an element beside the arena's
    23 a voxel).  A context with 8 MB beside a 64 MB arena has no room for it: the server opens all the same
    and serves in the Jacobi form."""
    solo, masks, ps = solo_and_requests()
    monkeypatch.setenv("FAST_TAU_RB_STAGED", "0")
    c = T.Context(0, 72 << 20)
    try:
        s = T.Server(c, hbm_budget=64 << 20, max_active=4)
        try:
            for r, q in zip(serve(s, masks, ps), solo):
                assert r.status == 0 and r.true_rel_residual <= 1e-9
                assert abs(r.tau - q.tau) <= 1e-6 * q.tau
        finally:
            s.close()
    finally:
        c.close()


def test_requests_that_leave_the_preconditioner_end_as_alone(monkeypatch):
    """With a limit of two iterations without a reliable update every request leaves the cycle, and the
    rounds are the Jacobi form's until one more is admitted: the solo results, bit for bit."""
    monkeypatch.setenv("FAST_TAU_MG_STALL", "2")
    solo, masks, ps = solo_and_requests()
    assert [r.restarts >= 1 for r in solo] == [True, True, False]
    c = T.Context(0)
    s = T.Server(c, hbm_budget=256 << 20, max_active=2)   # the third is admitted once another ends
    try:
        for r, q in zip(serve(s, masks, ps), solo):
            assert r.status == 0 and (r.tau, r.iterations, r.restarts) == (q.tau, q.iterations, q.restarts)
    finally:
        s.close()
        c.close()
