"""The launches over the coarse levels: extents whose levels are ragged against the tile of 32 x 10 cells,
odd in every axis, one cell thin, and several levels deep, alone and batched (where tiles of
different volumes share a launch and its planes per tile)."""
import numpy as np
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1

# (nx, ny, nz), direction; levels of more than 4096 cells run block-wise
SHAPES = [((126, 42, 38), 0), ((130, 78, 85), 2), ((66, 39, 85), 4), ((1, 400, 380), 3), ((2, 281, 262), 5),
          ((261, 1, 402), 1), ((193, 141, 122), 0)]


@pytest.mark.parametrize("shape,d", SHAPES, ids=[f"{s[0]}x{s[1]}x{s[2]}_{d}" for s, d in SHAPES])
def test_ragged_levels(ctx, shape, d):
    """As for the ragged shapes of the fine tiles: tau at a true residual of 1e-10 within 1e-7 of the
    FP64 CG's at 1e-12, in at most a third of its iterations (a wrong value on a level costs
    iterations, not accuracy)."""
    vol = ctx.volume(F.generate_ellipsoids(shape, 12.0, 0.35, 0.6, 5))
    ref, _ = vol.solve(T.make_params(d, CG, "double", 1e-12, 40000))
    res, _ = vol.solve(T.make_params(d, CG, "mixed", 1e-10, 40000))
    vol.close()
    assert ref.status == 0 and res.status == 0 and res.true_rel_residual <= 1e-10
    assert abs(res.tau - ref.tau) <= 1e-7 * ref.tau
    assert res.iterations <= ref.iterations // 3, (res.iterations, ref.iterations)


def test_batched_levels_give_the_solo_bits(ctx):
    vols = [ctx.volume(F.generate_ellipsoids(s, 12.0, 0.35, 0.6, 7 + i)) for i, (s, _) in enumerate(SHAPES)]
    ps = [T.make_params(d, CG, "mixed", 1e-9, 40000) for _, d in SHAPES]
    solo = [v.solve(p)[0] for v, p in zip(vols, ps)]
    for b, r in zip(T.solve_batch(ctx, vols, ps), solo):
        assert b.status == 0 and (b.tau, b.iterations, b.refinements) == (r.tau, r.iterations, r.refinements)
    for v in vols:
        v.close()
