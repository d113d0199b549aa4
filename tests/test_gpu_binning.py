"""Binning of small sets by one workgroup and of larger ones by ten launches:
grid, cells, order inside a cell and delimiters are the oracle's on both."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _points(n, kind):
    rng = np.random.default_rng(n)
    p = rng.random((n, 3))
    if kind == "one place":
        p[:] = [0.3, 0.4, 0.5]
    elif kind == "dense":  # three in four in one grid cell
        p[: 3 * n // 4] = 0.7 + 1e-6 * p[: 3 * n // 4]
    elif kind == "flat":
        p[:, 0] = 0.25
    return rng.permutation(p)


# 1, 4 and 12 points a thread, the last of each and one more; 16,384 cells and
# more (density 0.25, 0.9) go the general way
@pytest.mark.parametrize("n", [1, 2, 63, 1023, 1024, 1025, 4096, 4097, 10007, 12288, 12289, 16385])
@pytest.mark.parametrize("kind,density", [("uniform", 1.25), ("uniform", 0.25), ("uniform", 20.0), ("dense", 1.25),
                                          ("one place", 1.25), ("flat", 0.9)])
def test_small_sets(ctx, n, kind, density):
    pts = _points(n, kind)
    if kind == "one place" and n > 4097:
        pts = pts[:4097]  # every point of a cell looks at every other one
    d = tess.Diagram(ctx, pts, np.full(3, -0.1), np.full(3, 1.1), density=density,
                     groups=np.arange(len(pts)) % 5)
    d.query(tess.QUERY_CELLS, [[0.5, 0.5, 0.5]], 0.01)  # bins the points, computes no cell
    g, bins, srt, dl = orc.grid(pts, density)
    b, s, cpd = d.grid()
    assert cpd == g.cpd
    assert np.array_equal(b, [g.xmin, g.xmax, g.ymin, g.ymax, g.zmin, g.zmax])
    assert np.array_equal(s, [g.sx, g.sy, g.sz])
    cell, sorted_, delim = d.copy_grid()
    assert np.array_equal(cell, bins) and np.array_equal(sorted_, srt) and np.array_equal(delim, dl)
    # points and groups in grid order, through a query that returns them all
    off, ids = d.query(tess.QUERY_CLOUD, [[0.5, 0.5, 0.5]], np.inf, target_group=2)[:2]
    ro, ri = orc.queries(tess.QUERY_CLOUD, pts, [[0.5, 0.5, 0.5]], np.inf, density=density,
                         groups=np.arange(len(pts)) % 5, target_group=2)
    assert np.array_equal(off, ro) and np.array_equal(ids, ri)
    d.close()


# sets of up to 1 MiB (43,690 points) reach the device through one pinned
# buffer, one after the other: none may see the next one's points, and the
# caller's array is free once the call is back
@pytest.mark.parametrize("n", [1, 2, 3, 4, 43690, 43691])
def test_uploads_in_turn(ctx, n):
    sets = [np.random.default_rng(k).random((n, 3)) for k in range(6)]
    ds = []
    for p in sets:
        q = p.copy()
        ds.append(tess.Diagram(ctx, q, np.full(3, -0.1), np.full(3, 1.1), density=2.0))
        q[:] = 0.5
    for p, d in zip(sets, ds):
        d.query(tess.QUERY_CELLS, [[0.5, 0.5, 0.5]], 0.01)
        _, bins, srt, dl = orc.grid(p, 2.0)
        cell, sorted_, delim = d.copy_grid()
        assert np.array_equal(cell, bins) and np.array_equal(sorted_, srt) and np.array_equal(delim, dl)
        d.close()
