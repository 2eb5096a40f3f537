"""The row probe of kernels five cells wide against the oracle's pairs."""
import numpy as np
import pytest

from gpu_util import needs_gpu
from test_gpu_pairs import _subm

pytestmark = [pytest.mark.gpu, needs_gpu]


def _cells(seed, shape, B, n):
    rng = np.random.default_rng(seed)
    total = B * shape[0] * shape[1] * shape[2]
    keys = rng.choice(total, size=min(n, total), replace=False)
    x, r = keys % shape[2], keys // shape[2]
    y, r = r % shape[1], r // shape[1]
    return np.stack([r // shape[0], r % shape[0], y, x], 1).astype(np.int32)


@pytest.mark.parametrize("k,d", [(5, 1), ((1, 1, 5), 1), ((1, 5, 5), (1, 2, 1)), ((3, 2, 5), (3, 1, 1)),
                                 ((5, 5, 5), (2, 3, 1)), ((5, 5, 5), (1, 1, 2)), ((6, 5, 5), 1)])
def test_five_wide_kernels(k, d):
    """One kernel row to 25, rows in whole and partial batches of five, even
    extents and dilations in z and y; dil.x == 2 and more than 128 slots take
    the slot-by-slot probe.  Rows of cells at every x border and word straddle
    (a fully occupied 37-wide grid, grids narrower than the kernel), column
    counts around a block's 256, repeated coordinates, and a grid sparse
    enough for atomic marks (untouched tiles read as empty)."""
    full = np.stack(np.meshgrid(np.arange(2), np.arange(5), np.arange(6), np.arange(37),
                                indexing="ij"), -1).reshape(-1, 4).astype(np.int32)
    _subm(full[np.random.default_rng(0).permutation(len(full))], (5, 6, 37), 2, k, d, "full grid")
    for n in (1, 255, 256, 257):
        _subm(_cells(n, (9, 8, 11), 2, n), (9, 8, 11), 2, k, d, f"{n} columns")
    for w in (1, 2, 4, 33):
        _subm(_cells(w, (4, 4, w), 1, 12 * w), (4, 4, w), 1, k, d, f"{w} cells wide")
    rep = _cells(5, (7, 7, 70), 1, 900)
    _subm(np.concatenate([rep, rep[::3], rep[::7]]), (7, 7, 70), 1, k, d, "repeated rows")
    sparse = _cells(6, (41, 600, 700), 1, 3000)
    near = np.concatenate([sparse, np.clip(sparse + np.array([0, 1, -1, 2]), 0, [0, 40, 599, 699])])
    _subm(np.unique(near, axis=0).astype(np.int32), (41, 600, 700), 1, k, d, "atomic marks")
