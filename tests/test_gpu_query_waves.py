"""Box queries on both sides of the number up to which each gets a wavefront of
its own: few, 8,192 and one more, with short and long rows, against the oracle."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def _points(kind):
    rng = np.random.default_rng(5)
    if kind == "uniform":
        return rng.random((1500, 3))
    if kind == "dense":  # rows of hundreds of points beside empty ones
        return np.vstack([rng.random((300, 3)), 0.5 + 0.01 * rng.normal(size=(700, 3))])
    return rng.random((900, 3)) * [1, 1, 3.5e308] - [0, 0, 1.75e308]  # cells of infinite size along z


@pytest.mark.parametrize("nq", [1, 3, 4, 5, 64, 8191, 8192, 8193])
@pytest.mark.parametrize("points", ["uniform", "dense", "wide"])
@pytest.mark.parametrize("kind", [tess.QUERY_CELLS, tess.QUERY_CELL_RADIUS, tess.QUERY_REAL_RADIUS])
def test_few_and_many(ctx, nq, points, kind):
    rng = np.random.default_rng(nq)
    pts = _points(points)
    q = np.vstack([pts[rng.integers(0, len(pts), nq)], rng.uniform(-0.2, 1.2, (nq, 3))])[rng.permutation(2 * nq)[:nq]]
    # long walks for the few, now and then one for the many
    r = rng.choice([0.02, 0.05, -0.05, 0.4, np.inf, np.nan], nq, p=[.2, .2, .1, .2, .2, .1] if nq < 100 else
                   [.6, .36, .01, .01, .01, .01])
    d = tess.Diagram(ctx, pts, np.full(3, -1.79e308), np.full(3, 1.79e308), density=0.7)
    off, ids = d.query(kind, q, r)[:2]
    d.close()
    want_off, want = orc.queries(kind, pts, q, r, density=0.7)
    assert np.array_equal(off, want_off) and np.array_equal(ids, want)


# 64 boxes of 26,000 points take well under what 4,096 of them do (as long,
# where one wavefront walks four queries' rows one after the other)
def test_few_long_walks_time(ctx):
    pts = tess.clustered(200000, 2)
    d = tess.Diagram(ctx, pts, np.zeros(3), np.ones(3))
    r = tess.DeviceArray(ctx, np.array([0.2]))
    ms = {}
    for nq in (64, 4096):
        q = tess.DeviceArray(ctx, pts[np.random.default_rng(nq).integers(0, len(pts), nq)])
        fill = []
        for _ in range(9):
            h = d.query_device(tess.QUERY_REAL_RADIUS, q.ptr, nq, r.ptr, 1)
            fill.append(h.timings()["fill_ms"])
            h.close()
        ms[nq] = sorted(fill)[4]
    d.close()
    assert ms[64] < 0.85 * ms[4096], ms
