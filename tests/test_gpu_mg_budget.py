"""A device budget without room for what the multigrid preconditioner needs beside the solve's own vectors:
the solve is not refused, it takes the Jacobi form."""
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1


@pytest.mark.parametrize("staged", ["2", "0"])
def test_solve_within_the_budget_of_the_jacobi_form(monkeypatch, staged):
    """With one byte less than all allocations of a preconditioned solve (its own block, the last one,
    does not fit) a volume and a batch end at their tolerance with the same tau, in the Jacobi form's iterations."""
    monkeypatch.setenv("FAST_TAU_RB_STAGED", staged)
    masks = [F.generate_ellipsoids(s, 12.0, 0.35, 0.6, 4 + i) for i, s in enumerate([(64, 50, 48), (48, 50, 64)])]
    ps = [T.make_params(d, CG, "mixed", 1e-9, 20000) for d in (0, 4)]

    def run(budget, n):
        c = T.Context(0, budget)
        try:
            vols = [c.volume(m) for m in masks[:n]]
            return T.solve_batch(c, vols, ps[:n]), c.device_bytes()
        finally:
            c.close()

    for n in (1, 2):
        full, held = run(0, n)
        tight, tight_held = run(held - 1, n)
        assert tight_held < held
        for a, b in zip(full, tight):
            print(staged, n, a.iterations, b.iterations, a.tau, b.tau)
            assert a.status == 0 and b.status == 0 and b.true_rel_residual <= 1e-9
            assert b.iterations > 3 * a.iterations
            assert abs(a.tau - b.tau) <= 1e-6 * a.tau
