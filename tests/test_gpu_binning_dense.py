"""Small sets with dense grid cells: the order of cells below, at and above the
128 points from which they take turns in index order, up to all points in one."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _points(n, kind):
    rng = np.random.default_rng(n)
    p = rng.random((n, 3))
    if kind == "one cell":
        p[:] = [0.3, 0.4, 0.5]
    elif kind == "two cells":
        p[: n // 2] = 0.3 + 1e-7 * p[: n // 2]
        p[n // 2:] = 0.6 + 1e-7 * p[n // 2:]
        p[:2] = [[0, 0, 0], [1, 1, 1]]
    elif kind == "clusters":  # a hundred cells of about n / 100
        c = rng.random((100, 3))
        p = np.clip(c[rng.integers(0, 100, n)] + 1e-4 * rng.normal(size=(n, 3)), 0, 1)
    return p if kind == "in turn" else rng.permutation(p)


@pytest.mark.parametrize("n", [128, 129, 1023, 1024, 1025, 4096, 4097, 12287, 12288])
@pytest.mark.parametrize("kind,density", [("one cell", 1.25), ("two cells", 1.25), ("clusters", 1.25),
                                          ("uniform", 100.0), ("uniform", 115.0), ("uniform", 128.0), ("uniform", 900.0),
                                          ("in turn", 100.0)])
def test_dense_cells(ctx, n, kind, density):
    pts = _points(n, kind)
    d = tess.Diagram(ctx, pts, np.full(3, -0.1), np.full(3, 1.1), density=density)
    d.query(tess.QUERY_CELLS, [[0.5, 0.5, 0.5]], 0.01)  # bins the points, computes no cell
    _, bins, srt, dl = orc.grid(pts, density)
    cell, order, delim = d.copy_grid()
    assert np.array_equal(cell, bins) and np.array_equal(order, srt) and np.array_equal(delim, dl)
    # the points themselves in that order
    off, ids = d.query(tess.QUERY_REAL_RADIUS, pts[: min(n, 50)], 0.0)[:2]
    want_off, want = orc.queries(tess.QUERY_REAL_RADIUS, pts, pts[: min(n, 50)], 0.0, density=density)
    assert np.array_equal(off, want_off) and np.array_equal(ids, want)
    d.close()


# 12,000 points in ten clusters against as many spread out (twelve times as long
# where every point of a cell looks at every other one)
def test_dense_cells_time(ctx):
    rng = np.random.default_rng(1)
    c = rng.random((10, 3)) * 0.8 + 0.1
    clustered = np.clip(c[rng.integers(0, 10, 12000)] + 0.004 * rng.normal(size=(12000, 3)), 0, 1)
    ms = []
    for pts in (rng.random((12000, 3)), clustered):
        t = []
        for _ in range(9):
            d = tess.Diagram(ctx, pts, np.full(3, -0.1), np.full(3, 1.1))
            d.compute()
            t.append(d.timings()["bin_ms"])
            d.close()
        ms.append(sorted(t)[4])
    assert ms[1] < 4 * ms[0], ms
