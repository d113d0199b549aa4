"""A batch of more sets than one launch's grid y takes (65,536): every set's
shell table is built, and sets from all of the batch equal single diagrams."""
import numpy as np
import pytest

import tess

pytestmark = pytest.mark.gpu

FIELDS = ("volume", "face_count", "face_offset", "neighbor", "area")


def test_more_sets_than_grid_y(ctx):
    lo, hi = np.zeros(3), np.ones(3)
    # one to three points: tables of one offset, and (6 points) of 27
    sets = [(tess.uniform(6 if k % 1000 == 7 else 1 + k % 3, k), lo, hi) for k in range(66001)]
    b = tess.Batch(ctx, sets)
    b.compute()
    for k in [0, 1, 7, 32007, 32767, 32768, 32769, 65535, 65536, 65537, 65007, 66000]:
        d = tess.Diagram(ctx, *sets[k])
        d.compute()
        one, of_batch = d.cells(), b.cells(k)
        for f in FIELDS:
            assert np.array_equal(one[f], of_batch[f]), (k, f)
        d.close()
    b.close()
