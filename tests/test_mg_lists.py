"""The launch lists of the multigrid preconditioner, on the CPU: whatever volumes of a batch are still
unfinished when it is compacted, their lists fit into what was allocated for the whole batch."""
import ctypes as C

import numpy as np

from fast_amd import _lib


def blocks(dims, dirs, live):
    dims = np.ascontiguousarray(dims, np.int32)
    dirs = np.ascontiguousarray(dirs, np.int32)
    live = np.ascontiguousarray(live, np.uint8)
    out = (C.c_uint64 * 3)()
    rc = _lib.lib().fast_debug_mg_lists(len(dims), dims.ctypes.data_as(C.POINTER(C.c_int)),
                                        dirs.ctypes.data_as(C.POINTER(C.c_int)),
                                        live.ctypes.data_as(C.POINTER(C.c_uint8)), out)
    assert rc == _lib.FAST_OK
    return list(out)


# a batch whose tail has more blocks than the whole: fewer volumes take fewer planes per tile
BOXES = [(183, 199, 203), (183, 144, 150), (143, 184, 120), (152, 201, 119), (184, 204, 188), (200, 178, 193),
         (200, 148, 112), (135, 190, 124), (135, 200, 133), (159, 117, 102), (123, 108, 119), (189, 146, 204)]


def test_a_tail_with_more_blocks_than_the_batch_fits():
    room, whole, part = blocks(BOXES, [0] * len(BOXES), [i in (1, 2, 3, 5, 9, 11) for i in range(len(BOXES))])
    assert part > whole
    assert whole <= room and part <= room


def test_every_tail_fits():
    """Random batches over the sizes that take the cycle, thin and small volumes among them (the small
    ones have no lists), with several random sets of unfinished volumes each."""
    rng = np.random.default_rng(5)
    longer = 0
    for _ in range(300):
        n = int(rng.integers(2, 33))
        lo, hi = sorted(rng.integers(20, 260, 2))
        dims = rng.integers(lo, hi + 1, (n, 3))
        if rng.random() < 0.2:
            dims[rng.integers(n), rng.integers(3)] = rng.integers(1, 4)
        dirs = rng.integers(0, 6, n)
        for _ in range(4):
            room, whole, part = blocks(dims, dirs, rng.random(n) < rng.random())
            assert whole <= room and part <= room, (dims.tolist(), dirs.tolist())
            longer += part > whole
    assert longer > 0   # the sample holds tails that outgrow the batch's own lists
