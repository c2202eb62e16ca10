"""Stencil codes and labels at the row lengths where the four-voxel words of the code kernel end
(rows of 1 to 3 voxels, 4 k and the remainders), and labels of masks whose spans meet only across y
or z, against the oracle (whole numbers and the FP64 operator, whose sums have the oracle's
order: equal)."""
import numpy as np
import pytest

import fast_amd as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx", [1, 2, 3, 4, 5, 6, 7, 8, 63, 65, 258])
def test_codes_and_labels_by_row_length(ctx, nx):
    rng = np.random.default_rng(nx)
    for ny, nz in ((1, 1), (1, 6), (5, 1), (7, 9)):
        m = np.where(rng.random((nz, ny, nx)) < 0.4, rng.integers(1, 256, (nz, ny, nx)), 0).astype(np.uint8)
        vol = ctx.volume(m)
        assert vol.count_zero() == int((m == 0).sum())
        x = rng.standard_normal(m.shape)
        for d in (0, 3, 4):
            assert np.array_equal(vol.apply(d, x), O.apply(m, d, x)), (m.shape, d)
        vol.close()
        b = np.where(m > 0, 255, 0).astype(np.uint8)
        vol = ctx.volume(b)
        lab, nl = vol.ccl_labels(255)
        olab, onl = O.ccl(b)
        assert nl == onl and np.array_equal(lab, olab), m.shape
        vol.close()


def test_labels_of_a_winding_path(ctx):
    """One pore path through every second plane, joined by single voxels at alternating ends: the links
    across z stand alone, with solid all around."""
    m = np.full((41, 23, 70), 255, np.uint8)
    m[::2] = 0
    m[::2, 1::4, 1:] = 255
    m[::2, 3::4, :-1] = 255
    m[1::4, -1, -1] = 0
    m[3::4, 0, 0] = 0
    vol = ctx.volume(m)
    lab, nl = vol.ccl_labels(255)
    olab, onl = O.ccl(m)
    assert nl == onl and np.array_equal(lab, olab)
    vol.close()
