"""Cells that are tested against thousands of candidates which do not cut them:
points on a sphere, every one a neighbour candidate of every other."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)


def _sphere(n):
    p = np.random.default_rng(1).normal(size=(n, 3))
    return p / np.linalg.norm(p, axis=1)[:, None] * 0.45 + 0.5


@pytest.mark.parametrize("capacity", [64, 128, 256])
def test_cells_of_a_sphere(ctx, capacity):
    pts = _sphere(900)
    d = tess.Diagram(ctx, pts, LO, HI, vertex_capacity=capacity, collect_stats=True)
    d.compute()
    got, stats = d.cells(), d.stats()
    ref = orc.compute(pts, LO, HI)
    for f in ("face_count", "face_offset", "neighbor"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    for f in ("classified", "cuts", "flops"):
        assert np.array_equal(stats[f], ref["stats"][f]), f
    d.close()


# Both passes are bound by the instructions of their tests and cuts: 20,000
# cells of 20,000 tests each take 19 times as long as 300,000 cells of spread
# out points, 27 times when vertices that were cut off still count in the
# pre-test of a chunk.
def test_time_of_a_sphere(ctx):
    ms = []
    for pts in (tess.uniform(300000, 1), _sphere(20000)):
        d = tess.Diagram(ctx, pts, LO, HI)
        t = []
        for _ in range(5):
            d.compute_status()  # (a few cells of the sphere fail their topology checks)
            t.append(d.timings()["cells_ms"])
        ms.append(sorted(t)[2])
        d.close()
    assert ms[1] < 23 * ms[0], ms
