"""Tile shapes of the full-grid passes, on the CPU: the rule against a plain restatement, and its time on
volumes that are very long in z."""
import ctypes as C
import time

import numpy as np
import pytest

from fast_amd import _lib

FP64, FP32, MIXED = 0, 1, 2


def shape(dims, precision):
    dims = np.ascontiguousarray(dims, np.int32)
    out = (C.c_int * 3)()
    assert _lib.lib().fast_debug_tile_shape(len(dims), dims.ctypes.data_as(C.POINTER(C.c_int)), precision, out) == 0
    return tuple(out)


def up(a, b):
    return -(-a // b)


def plain(dims, precision, shapes=None):
    """The least modelled time over every number of tiles along z; a batch of more than two rounds
    chooses again among the shapes that cost least traffic."""
    order = ([(64, 16), (64, 8), (32, 32), (32, 16), (64, 4), (32, 8), (16, 16)] if precision == FP64 else
             [(64, 8), (64, 16), (32, 16), (32, 32), (64, 4), (32, 8), (16, 16)])
    held, prologue, keeps_up = (24 if precision == FP32 else 16), (1 if precision == FP64 else 2), (12 if precision == FP64 else 18)
    nz = max(d[2] for d in dims)
    best = None
    for tx, ty, weight in [(x, y, 1.0) for x, y in order] if shapes is None else shapes:
        waves = tx * ty // 64
        cap, last = 256 * (held // waves), 0
        for n in range(1, nz + 1):
            tz = up(nz, n)
            if tz == last or tz > 64 or (tz < 2 and nz > 1):
                continue
            last = tz
            tiles = sum(up(x, tx) * up(y, ty) * up(z, tz) for x, y, z in dims)
            full, rest = divmod(tiles, cap)
            t = (tz + prologue) * weight * (full * max(1.0, held // waves * waves / keeps_up) +
                                            (max(1.0, up(rest, 256) * waves / keeps_up) if rest else 0.0))
            if best is None or t < best[0]:
                best = (t, (tx, ty, tz), tiles / cap)
    if shapes is None and len(dims) > 1 and best[2] > 2:
        return plain(dims, precision, [(64, 8, 1.0), (64, 4, 1.0), (32, 8, 1.1)])
    return best[1]


@pytest.mark.parametrize("precision", [FP64, FP32, MIXED])
def test_the_rule_is_the_plain_one(precision):
    rng = np.random.default_rng(precision)
    for _ in range(60):
        d = [tuple(int(v) for v in np.exp(rng.uniform(0, np.log(400), 3)).round())]
        assert shape(d, precision) == plain(d, precision), d
    assert shape([(1, 1, 1)], precision)[2] == 1


@pytest.mark.parametrize("precision", [FP64, FP32, MIXED])
def test_batches_of_many_rounds_take_wide_blocks(precision):
    """Random batches take the plain rule's shape; one that runs many rounds never the 16 x 16 blocks whose
    halo made it 15-20% slower."""
    rng = np.random.default_rng(10 + precision)
    many = [tuple(int(v) for v in rng.integers(100, 161, 3)) for _ in range(10)]
    assert shape(many, precision)[0] >= 32
    for _ in range(40):
        lo, hi = sorted(int(v) for v in rng.integers(16, 200, 2))
        d = [tuple(int(v) for v in rng.integers(lo, hi + 1, 3)) for _ in range(int(rng.integers(2, 20)))]
        assert shape(d, precision) == plain(d, precision), d


def test_long_volumes_take_no_time():
    """2^29 voxels, all along z, are chosen for in well under a millisecond of host time per call (a loop
    over the tiles along z took seconds)."""
    t = time.perf_counter()
    for _ in range(10):
        s = shape([(1, 1, (1 << 29) - 1)], FP64)
    assert time.perf_counter() - t < 0.1
    assert 2 <= s[2] <= 64


def test_large_batches_have_finalize_launches():
    """A volume's finalizes are folded up to its tile limit, and a batch's only up to 2048 tiles in all."""
    def folds(tiles, precision):
        return _lib.lib().fast_debug_folds(len(tiles), (C.c_int * len(tiles))(*tiles), precision)

    assert [folds([n], FP64) for n in (1, 1100, 1101)] == [1, 1, 0]
    assert [folds([n], FP32) for n in (1, 512, 513)] == [1, 1, 0]
    for precision in (FP64, FP32):
        assert folds([256] * 8, precision) == 1 and folds([256] * 8 + [1], precision) == 0
        assert folds([324] * 9 + [55], precision) == 0
