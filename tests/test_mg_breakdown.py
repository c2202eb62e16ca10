"""The scalar recurrence of the preconditioned CG, on the CPU: every way in which the multigrid cycle can
fail leads to the Jacobi form, which keeps its whole iteration cap.  The system's diagonal is negative, and so are
r.z and p.q while all is well."""
import ctypes as C

import pytest

from fast_amd import _lib

UPDATE, CYCLE, PQ, END = 0, 1, 2, 3          # events of fast_debug_cg_state
INF, NAN = float("inf"), float("nan")


def run(events, mg=1, tol=1e-9, max_iter=1000):
    """(status, mg, iterations, updates) after each event."""
    n = len(events)
    ev = (C.c_int * n)(*[e for e, _ in events])
    val = (C.c_double * n)(*[v for _, v in events])
    out = (C.c_int64 * (4 * n))()
    assert _lib.lib().fast_debug_cg_state(mg, tol, max_iter, n, ev, val, out) == _lib.FAST_OK
    return [tuple(out[4 * i:4 * i + 4]) for i in range(n)]


START = [(UPDATE, 1.0)]
IT = [(CYCLE, -1.0), (PQ, -1.0), (END, 0.5)]   # an ordinary iteration: no update is due


def status(name):
    """Status numbers, taken from the recurrence: a volume runs after its first update, and is fresh
    again after a residual that is not finite."""
    return {"running": run(START)[-1][0], "fresh": run(START + [(PQ, -1.0), (END, NAN)], mg=0)[-1][0]}[name]


FAILURES = {"growth": [(CYCLE, -1.0), (PQ, -1.0), (END, 1.1e4)], "residual": [(CYCLE, -1.0), (PQ, -1.0), (END, NAN)],
            "alpha": [(CYCLE, -1.0), (PQ, 0.0)], "alpha_nan": [(CYCLE, -1.0), (PQ, NAN)],
            "rz_positive": [(CYCLE, 1.0)], "rz_zero": [(CYCLE, 0.0)], "rz_nan": [(CYCLE, NAN)], "rz_inf": [(CYCLE, -INF)]}


@pytest.mark.parametrize("name", FAILURES)
def test_breakdown_leaves_the_cycle(name):
    """After a breakdown the volume starts afresh without the cycle, which on the same residual would
    break down again, and counts its iterations anew."""
    out = run(START + 9 * IT + FAILURES[name] + [(UPDATE, 1.0)] + 3 * [(PQ, -1.0), (END, 0.5)])
    fail = out[len(START) + 9 * len(IT) + len(FAILURES[name]) - 1]
    assert out[len(START) + 9 * len(IT) - 1] == (status("running"), 1, 9, 1)
    assert fail[:3] == (status("fresh"), 0, 0)
    assert out[-7][:2] == (status("running"), 0) and out[-1] == (status("running"), 0, 3, 2)


def test_stall_leaves_the_cycle():
    out = run(START + 128 * IT)
    assert out[3 * 127][:3] == (status("running"), 1, 127) and out[-1][:3] == (status("fresh"), 0, 0)


def test_the_jacobi_form_keeps_its_cap():
    """A cap of 12 that nine iterations of a failing cycle have used up in part still leaves 12 from the
    cycle's x64, and after those 12 from x0 (no updates counted); then the volume ends."""
    jacobi = 12 * [(PQ, -1.0), (END, 0.5)] + START
    out = run(START + 9 * IT + FAILURES["growth"] + START + jacobi + START + jacobi, max_iter=12)
    first, second = out[-26 - len(jacobi):-len(jacobi)], out[-len(jacobi) - 1:]
    assert [o[2] for o in first[:24:2]] == list(range(0, 12)) and first[-2][:3] == (status("fresh"), 0, 0)
    assert first[-2][3] == 0 and second[0] == (status("running"), 0, 0, 1)
    assert second[-1][2] == 12 and second[-1][0] not in (status("running"), status("fresh"))


@pytest.mark.parametrize("fail", [[(PQ, -1.0), (END, 1.1e4)], [(PQ, 0.0)]], ids=["growth", "alpha"])
def test_a_second_breakdown_starts_from_x0(fail):
    """Where the Jacobi form breaks down from the cycle's x64 as well it starts from x0, as a solve without
    the cycle does; from there on a breakdown is a fresh start that keeps the count."""
    begin = START + 3 * IT + FAILURES["residual"] + START
    out = run(begin + 2 * [(PQ, -1.0), (END, 0.5)] + fail + START + [(PQ, -1.0), (END, 0.5)] + fail)
    again = len(begin) + 4 + len(fail)
    assert out[again - 1] == (status("fresh"), 0, 0, 0) and out[again] == (status("running"), 0, 0, 1)
    assert out[-1] == (status("fresh"), 0, len(fail), 1)


def test_slow_after_a_breakdown_starts_from_x0():
    """1024 iterations without a reliable update from the x64 of a cycle that broke down; after one that was
    only slow the Jacobi form keeps its cap."""
    slow = [(PQ, -1.0), (END, 0.5)]
    broke = run(START + 3 * IT + FAILURES["growth"] + START + 1024 * slow, max_iter=5000)
    assert broke[-3][2] == 1023 and broke[-1] == (status("fresh"), 0, 0, 0)
    stalled = run(START + 128 * IT + START + 2000 * slow, max_iter=5000)
    assert stalled[-1][:3] == (status("running"), 0, 2000)


def test_a_residual_that_is_not_finite_starts_from_x0():
    out = run(START + 3 * IT + [(CYCLE, -1.0), (PQ, -1.0), (END, 1e-4), (UPDATE, NAN)] + START)
    assert out[-2] == (status("fresh"), 0, 0, 0) and out[-1] == (status("running"), 0, 0, 1)
    assert run([(UPDATE, NAN)])[-1][0] not in (status("running"), status("fresh"))   # the system's own


@pytest.mark.parametrize("fail", [[(PQ, -1.0), (END, 1.1e4)], [(PQ, 0.0)]], ids=["growth", "alpha"])
def test_the_jacobi_form_starts_afresh_as_ever(fail):
    """Without the cycle a breakdown is a fresh start that keeps the count."""
    out = run(START + 4 * [(PQ, -1.0), (END, 0.5)] + fail, mg=0)
    assert out[-1][:3] == (status("fresh"), 0, 4 + (len(fail) - 1))
