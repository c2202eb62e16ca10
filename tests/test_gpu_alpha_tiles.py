"""The area kernel's tiles: 4, 8 or 16 planes by the size of the volume, ragged on every axis, with
0/255 bytes (interpolation parameters from a table), arbitrary bytes (divisions) and both in one wave.

The oracle rounds each cube's sum of areas to double, the kernel sums all triangles in double-double:
the up to five float areas of a cube of 0/255 corners add up without rounding, so the totals are
equal; otherwise a cube's sum is off by at most half an ulp of itself and the total, rounded once
on either side, by at most two ulps."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (nz, ny, nx): below 2048, below 8192 and above 8192 tiles of 64 x 4 x 16
SHAPES = [(9, 6, 65), (5, 9, 129), (529, 258, 3), (1013, 517, 2)]


@pytest.mark.parametrize("shape", SHAPES)
def test_area_of_binary_and_mixed_bytes(ctx, shape):
    rng = np.random.default_rng(sum(shape))
    m = np.where(rng.random(shape) < 0.45, 255, 0).astype(np.uint8)
    vol = ctx.volume(m)
    assert vol.area() == O.mc_area(m)
    assert np.array_equal(vol.area_tensor(), O.mc_area_tensor(m))
    vol.close()
    gray = rng.random(shape) < 0.02
    m[gray] = rng.integers(0, 256, size=int(gray.sum()), dtype=np.uint8)
    vol = ctx.volume(m)
    for iso in (0.5, 0.31):
        a, ref = vol.area(iso), O.mc_area(m, iso)
        assert abs(a - ref) <= 2 * np.spacing(ref), (iso, a, ref)
    vol.close()
