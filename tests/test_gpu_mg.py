"""The multigrid preconditioner of the mixed CG: the same solution as the converged FP64 solve on
extents at the edges of its tiles, coarse cells and rules, the same bits whatever launches it."""
import numpy as np
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1

# (nx, ny, nz), direction: fine tiles are 64 slots (128 voxels) x 8 rows x an even number of planes,
# coarse cells 2 x 2 x 2; 98304 voxels and 24 voxels along the flow are the smallest that take it
SHAPES = [((96, 32, 32), 0), ((48, 46, 45), 2), ((129, 33, 31), 4), ((127, 40, 41), 1), ((131, 65, 63), 3),
          ((257, 24, 17), 2), ((24, 97, 95), 0), ((130, 73, 25), 5), ((3, 300, 120), 2), ((300, 1, 400), 4),
          ((17, 16, 401), 4), ((1000, 11, 9), 0)]


@pytest.mark.parametrize("shape,d", SHAPES, ids=[f"{s[0]}x{s[1]}x{s[2]}_{d}" for s, d in SHAPES])
def test_matches_converged_fp64(ctx, shape, d):
    """At a true residual of 1e-10 tau is within 1e-7 of the FP64 CG's at 1e-12 (whose recurrences
    are the oracle's) and the field within 1e-6, in a fraction of the iterations: the same bars per
    residual as the Jacobi form's on ragged shapes."""
    m = F.generate_ellipsoids(shape, 12.0, 0.35, 0.6, 5)
    vol = ctx.volume(m)
    ref, cref = vol.solve(T.make_params(d, CG, "double", 1e-12, 40000), conc=True)
    res, c = vol.solve(T.make_params(d, CG, "mixed", 1e-10, 40000), conc=True)
    vol.close()
    err, dc = abs(res.tau - ref.tau) / ref.tau, np.abs(c - cref).max()
    print(f"{shape} d={d}: it={res.iterations} (FP64 CG {ref.iterations}) err={err:.1e} max|dc|={dc:.1e}")
    assert ref.status == 0 and res.status == 0 and res.true_rel_residual <= 1e-10
    assert err <= 1e-7 and dc <= 1e-6
    assert res.iterations <= ref.iterations // 3


@pytest.mark.parametrize("coeffs", [(1.0, 1e-5), (0.001, 1.0), (1.0, 1.0)])
def test_other_conductivities(ctx, coeffs):
    m = F.generate_ellipsoids((70, 61, 52), 12.0, 0.5, 0.6, 2)
    vol = ctx.volume(m)
    for d in (1, 4):
        ref, _ = vol.solve(T.make_params(d, CG, "double", 1e-13, 40000, coeffs))
        res, _ = vol.solve(T.make_params(d, CG, "mixed", 1e-10, 40000, coeffs))
        assert ref.status == 0 and res.status == 0
        assert abs(res.tau - ref.tau) <= 1e-6 * ref.tau, (coeffs, d, res.tau, ref.tau)
    vol.close()


def test_forms_tiles_and_batches_give_the_same_bits(ctx, monkeypatch):
    """The separate and fused Y and Q passes, other red-black tiles, and a batch with volumes of the
    Jacobi form (which end much later) give the solo result bit for bit."""
    masks = [F.generate_ellipsoids(s, 12.0, 0.35, 0.6, 3 + i)
             for i, s in enumerate([(66, 51, 47), (40, 40, 40), (129, 31, 33), (200, 200, 12)])]
    dirs = [0, 2, 5, 4]
    vols = [ctx.volume(m) for m in masks]
    ps = [T.make_params(d, CG, "mixed", 1e-9, 40000) for d in dirs]
    solo = [v.solve(p, conc=True) for v, p in zip(vols, ps)]
    for b, (r, _) in zip(T.solve_batch(ctx, vols, ps), solo):
        assert b.status == 0 and (b.tau, b.iterations, b.refinements) == (r.tau, r.iterations, r.refinements)
    for mode in ("0", "1"):
        monkeypatch.setenv("FAST_TAU_RB_STAGED", mode)
        got, c = vols[0].solve(ps[0], conc=True)
        monkeypatch.delenv("FAST_TAU_RB_STAGED")
        assert got.iterations == solo[0][0].iterations and np.array_equal(c, solo[0][1])
    ctx.set_rb_shape(9, 7, 3)
    got, c = vols[2].solve(ps[2], conc=True)
    ctx.set_rb_shape(0)
    assert got.iterations == solo[2][0].iterations and np.array_equal(c, solo[2][1])
    for v in vols:
        v.close()


def test_stalled_volume_goes_on_with_the_jacobi_form(monkeypatch):
    """With a limit of two iterations without a reliable update every solve changes over to the
    Jacobi form from its x64 and still ends below its tolerance, alone and in a batch."""
    monkeypatch.setenv("FAST_TAU_MG_STALL", "2")
    c = T.Context(0)
    try:
        vols = [c.volume(F.generate_ellipsoids(s, 12.0, 0.35, 0.6, 9)) for s in ((64, 50, 48), (48, 50, 64), (40, 30, 30))]
        ps = [T.make_params(d, CG, "mixed", 1e-9, 30000) for d in (0, 4, 2)]
        solo = [v.solve(p)[0] for v, p in zip(vols, ps)]
        ref = [v.solve(T.make_params(d, CG, "double", 1e-12, 30000))[0] for v, d in zip(vols, (0, 4, 2))]
        for b, r, f in zip(T.solve_batch(c, vols, ps), solo, ref):
            assert b.status == 0 and (b.tau, b.iterations) == (r.tau, r.iterations)
            assert r.true_rel_residual <= 1e-9 and abs(r.tau - f.tau) <= 1e-6 * f.tau
        assert [r.restarts >= 1 for r in solo] == [True, True, False]
    finally:
        c.close()
