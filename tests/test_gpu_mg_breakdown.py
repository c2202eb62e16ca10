"""Solid conductivities at which the FP32 multigrid cycle breaks down on the way to a small residual: the
solve goes on with the Jacobi form and ends at its tolerance, alone and in a batch."""
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1

# (nx, ny, nz), semi-axis ratio, solid fraction, direction, solid conductivity
CASES = [((48, 46, 45), 0.35, 0.75, 2, 1e-8), ((48, 46, 45), 0.35, 0.75, 2, 1e-7), ((100, 101, 97), 0.35, 0.65, 4, 1e-7),
         ((128, 128, 128), 5.0, 0.75, 2, 1e-8)]


def test_breakdown_ends_in_a_converged_solve(ctx):
    """Residual 1e-9 within 3000 iterations of the Jacobi form (which takes 876 to 2089 of them by itself),
    tau within 1e-5 of the FP64 CG's at 1e-11; a batch gives the solo bits."""
    vols = [ctx.volume(F.generate_ellipsoids(s, 12.0, r, solid, 5)) for s, r, solid, _, _ in CASES]
    ps = [T.make_params(d, CG, "mixed", 1e-9, 3000, (1.0, ds)) for _, _, _, d, ds in CASES]
    solo = [v.solve(p)[0] for v, p in zip(vols, ps)]
    for v, r, (s, _, _, d, ds) in zip(vols, solo, CASES):
        ref, _ = v.solve(T.make_params(d, CG, "double", 1e-11, 40000, (1.0, ds)))
        print(s, ds, "it", r.iterations, "restarts", r.restarts, "tau", r.tau, "FP64", ref.tau, ref.iterations)
        assert r.status == 0 and r.true_rel_residual <= 1e-9 and ref.status == 0
        assert abs(r.tau - ref.tau) <= 1e-5 * ref.tau
    assert any(r.restarts for r in solo)   # the cycle did break down
    for b, r in zip(T.solve_batch(ctx, vols, ps), solo):
        assert b.status == 0 and (b.tau, b.iterations, b.refinements) == (r.tau, r.iterations, r.refinements)
    for v in vols:
        v.close()


def test_a_solve_that_is_stuck_after_the_breakdown_starts_from_x0(ctx):
    """Volumes on which the Jacobi form converges from x0 (in 2465, 1845 and 1177 iterations) and not from what
    the cycle left."""
    restarts = []
    for shape, solid, seed, d, ds, tol in (((48, 46, 45), 0.75, 6, 2, 1e-8, 1e-9), ((48, 46, 45), 0.75, 7, 2, 1e-8, 1e-9),
                                           ((80, 60, 40), 0.7, 6, 0, 1e-9, 1e-10)):
        vol = ctx.volume(F.generate_ellipsoids(shape, 12.0, 0.35, solid, seed))
        res, _ = vol.solve(T.make_params(d, CG, "mixed", tol, 4000, (1.0, ds)))
        ref, _ = vol.solve(T.make_params(d, CG, "double", 1e-11, 40000, (1.0, ds)))
        vol.close()
        print(shape, seed, res.iterations, res.restarts, res.tau, ref.tau, ref.iterations)
        assert res.status == 0 and res.true_rel_residual <= tol
        assert ref.status == 0 and abs(res.tau - ref.tau) <= 1e-5 * ref.tau
        restarts.append(res.restarts)
    assert max(restarts) >= 2
