"""Finalizes folded into the next pass: any round length, a batch whose volumes end at different
iterations, and volumes on either side of the tile limit give the oracle's iterations and tau."""
import numpy as np
import pytest

import fast_amd as F
from fast_amd import tau as T
from fast_amd._lib import lib
from oracle import oracle as O

pytestmark = pytest.mark.gpu
BICG, CG = 0, 1


@pytest.mark.parametrize("prec", ["double", "float"])
@pytest.mark.parametrize("solver", [CG, BICG])
def test_round_lengths_and_batches_equal_the_oracle(ctx, solver, prec):
    shapes = [((9, 7, 12), 0), ((33, 20, 17), 3), ((1, 1, 5), 4), ((50, 31, 48), 5)]
    masks = [F.generate_ellipsoids(s, 6.0, 0.5, 0.5, 11 + i) for i, (s, _) in enumerate(shapes)]
    refs = [O.tau(m, d, solver=solver, precision=int(prec == "float"), tol=1e-5)[0] for m, (_, d) in zip(masks, shapes)]
    vols = [ctx.volume(m) for m in masks]
    ps = [T.make_params(d, solver, prec, 1e-5, 10000) for _, d in shapes]
    try:
        for rnd in (1, 2, 3, 5, 16):
            assert lib().fast_ctx_set_round(ctx.handle, rnd) == 0
            for got in (T.solve_batch(ctx, vols, ps), [v.solve(p)[0] for v, p in zip(vols, ps)]):
                for r, q in zip(got, refs):
                    same = r.tau == q.tau or (np.isinf(r.tau) and np.isinf(q.tau)) or (np.isnan(r.tau) and np.isnan(q.tau))
                    assert r.iterations == q.iterations and same, (solver, prec, rnd, r.tau, q.tau)
    finally:
        lib().fast_ctx_set_round(ctx.handle, 0)
        for v in vols:
            v.close()


@pytest.mark.parametrize("tz", [2, 8])
def test_volumes_around_the_tile_limit_equal_the_oracle(ctx, tz):
    """16 x 16 tiles of 2 planes: 100 x 60 x 96 has 1344 tiles (finalize launches), of 8 planes 336
    (folded); both solvers take the oracle's path."""
    m = F.generate_ellipsoids((100, 60, 96), 8.0, 0.5, 0.4, 3)
    vol = ctx.volume(m)
    assert lib().fast_ctx_set_tile_shape(ctx.handle, 16, 16, tz) == 0
    try:
        for solver in (CG, BICG):
            ref, _ = O.tau(m, 2, solver=solver, tol=1e-3)
            res, _ = vol.solve(T.make_params(2, solver, "double", 1e-3, 10000))
            assert res.iterations == ref.iterations and res.tau == ref.tau
    finally:
        lib().fast_ctx_set_tile_shape(ctx.handle, 0, 0, 0)
        vol.close()
