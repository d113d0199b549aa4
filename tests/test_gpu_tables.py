"""Shell tables built on the device: the search walks them in canonical order,
so cells and their counters equal the oracle's for every grid shape."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _points(cells, scale, flat):
    # `cells` grid cells per dimension at 1.25 points per cell
    n = max(1, int(1.25 * cells**3) - 1) if cells > 1 else 1
    pts = np.random.default_rng(cells).random((n, 3))
    pts[:, 2] = 0.5 if flat else pts[:, 2]
    return pts * scale


# grids of 1 to 3 cells, both sides of the default table's 12 rings, and one
# well past it; equal sizes (many equal keys), ratios that make keys of
# different gaps equal, and sizes apart
@pytest.mark.parametrize("cells", [1, 2, 3, 12, 13, 14, 20])
@pytest.mark.parametrize("scale", [(1.0, 1.0, 1.0), (1.0, 2.0, 0.5), (1.0, 0.37, 0.02)])
def test_cells_for_grid_shapes(ctx, cells, scale):
    pts = _points(cells, np.array(scale), False)
    if cells > 2:  # the corners: cell sizes are exactly scale / cells apart by these ratios
        pts[0], pts[1] = 0.0, scale
    lo, hi = -0.05 * np.array(scale), 1.05 * np.array(scale)
    d = tess.Diagram(ctx, pts, lo, hi, collect_stats=True)
    d.compute()
    got, st = d.cells(), d.stats()
    ref = orc.compute(pts, lo, hi)
    for f in ("face_count", "face_offset", "neighbor"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    assert np.allclose(got["area"], ref["area"], rtol=1e-12, atol=0)
    for f in set(st.dtype.names) & set(ref["stats"].dtype.names) - {"status"}:
        assert np.array_equal(st[f], ref["stats"][f]), f
    d.close()


# every set of a batch has a table of its own, a flat one among them
def test_tables_of_a_batch(ctx):
    shapes = [(1, (1, 1, 1), False), (3, (1, 1, 1), False), (13, (1, 2, 0.5), False), (14, (1, 0.3, 0.1), False),
              (9, (1, 1, 1), True), (20, (1, 1, 1), False)]
    sets = []
    for cells, scale, flat in shapes:
        s = np.array(scale, float)
        sets.append((_points(cells, s, flat), -0.05 * s, 1.05 * s))
    b = tess.Batch(ctx, sets)
    b.compute()
    for k, (pts, lo, hi) in enumerate(sets):
        ref, got = orc.compute(pts, lo, hi), b.cells(k)
        for f in ("face_count", "face_offset", "neighbor"):
            assert np.array_equal(got[f], ref[f]), (k, f)
        assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    b.close()
