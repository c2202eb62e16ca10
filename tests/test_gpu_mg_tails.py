"""Tails of preconditioned batches: once the unfinished volumes hold at most half of the launched tiles
the launch lists are made anew for them, here with more coarse-level blocks than the whole batch's."""
import numpy as np
import pytest

import fast_amd as F
from fast_amd import tau as T

pytestmark = pytest.mark.gpu
CG = 1

# volumes (of those in test_mg_lists.py, whose lists they make) that are still unfinished when the batch is compacted
BOXES = [(183, 199, 203), (183, 144, 150), (143, 184, 120), (152, 201, 119), (184, 204, 188), (200, 178, 193),
         (200, 148, 112), (135, 190, 124), (135, 200, 133), (159, 117, 102), (123, 108, 119), (189, 146, 204)]
SLOW = (1, 2, 3, 5, 9, 11)


def test_compacted_preconditioned_batch_equals_solo(ctx):
    """Six empty volumes end several polling rounds before six porous ones; every result is that of
    the volume alone, bit for bit."""
    vols = [ctx.volume(F.generate_ellipsoids(b, 12.0, 5.0, 0.7, 20 + i) if i in SLOW
                       else np.zeros((b[2], b[1], b[0]), np.uint8)) for i, b in enumerate(BOXES)]
    p = T.make_params(0, CG, "mixed", 1e-9, 20000)
    solo = [v.solve(p)[0] for v in vols]
    its = [r.iterations for r in solo]
    print(its)
    assert min(its[i] for i in SLOW) > max(n for i, n in enumerate(its) if i not in SLOW) + 8   # two polling rounds
    for b, r in zip(T.solve_batch(ctx, vols, [p] * len(vols)), solo):
        assert b.status == 0 and (b.tau, b.iterations, b.refinements) == (r.tau, r.iterations, r.refinements)
    for v in vols:
        v.close()
