"""Box queries over grids whose extent along an axis is past the largest
double: the size of a grid cell is then infinite, a gap of 0 cells no number,
and the cells a radius reaches need not be neighbours along z."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

WIDE = 3.5e308  # (max - min) overflows, the coordinates do not


# z wide (rows are no intervals), x wide (they are), all wide, none
@pytest.mark.parametrize("wide", [(0, 0, 1), (1, 0, 0), (1, 1, 1), (0, 0, 0)])
# a few queries, and enough of them to be taken in grid order
@pytest.mark.parametrize("nq", [7, 4099])
@pytest.mark.parametrize("kind", [tess.QUERY_CELLS, tess.QUERY_CELL_RADIUS, tess.QUERY_REAL_RADIUS])
def test_wide_extents(ctx, wide, nq, kind):
    rng = np.random.default_rng(nq)
    u = rng.random((300, 3))
    w = np.array(wide, bool)
    pts = np.where(w, (u - 0.5) * WIDE, u)
    q = np.where(w, (rng.random((nq, 3)) - 0.5) * WIDE, rng.random((nq, 3)))
    r = rng.choice([0.0, 0.3, 1e307, -0.2, np.inf, -np.inf, np.nan], nq)
    r[:7] = [0.0, 0.3, 1e307, -0.2, np.inf, -np.inf, np.nan]
    d = tess.Diagram(ctx, pts, np.full(3, -1.79e308), np.full(3, 1.79e308), density=2.0)
    off, ids = d.query(kind, q, r)[:2]
    d.close()
    want_off, want = orc.queries(kind, pts, q, r, density=2.0)
    assert np.array_equal(off, want_off) and np.array_equal(ids, want)
