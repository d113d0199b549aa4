"""Scans by one workgroup and by three launches, and the reruns of sites that
outgrow a capacity, at the sizes where the route changes."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)


# one workgroup scans 4,096 counts at a time and up to 16,384: of points (face
# offsets) and of grid cells (15,625 = 25^3 and 17,576 = 26^3)
@pytest.mark.parametrize("n,density", [(1, 1.25), (4095, 1.25), (4096, 1.25), (4097, 1.25), (16384, 1.25),
                                       (16385, 1.25), (19000, 1.25), (20600, 1.25), (22000, 1.25)])
def test_offsets_and_delimiters(ctx, n, density):
    pts = tess.uniform(n, n + 1)
    d = tess.Diagram(ctx, pts, LO, HI, density=density)
    d.compute()
    got = d.cells()
    assert got["face_offset"][0] == 0
    assert np.array_equal(np.diff(got["face_offset"].astype(np.int64)), got["face_count"].astype(np.int64))
    g, bins, srt, dl = orc.grid(pts, density)
    cell, sorted_, delim = d.copy_grid()
    assert np.array_equal(cell, bins) and np.array_equal(sorted_, srt) and np.array_equal(delim, dl)
    ref = orc.compute(pts, LO, HI, density=density)
    assert np.array_equal(got["face_offset"], ref["face_offset"])
    assert np.array_equal(got["neighbor"], ref["neighbor"])
    d.close()


# points on a sphere of radius 0.45: cells of sites near its centre have about
# 2 (n - 2) vertices, below 64, 128 and 256 and past them
@pytest.mark.parametrize("capacity", [0, 128, 256])
@pytest.mark.parametrize("n", [30, 34, 60, 70, 120, 140])
def test_sites_by_capacity(ctx, n, capacity):
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3))
    pts = p / np.linalg.norm(p, axis=1)[:, None] * 0.45 + 0.5
    sites = np.vstack([0.5 + 0.01 * rng.normal(size=(20, 3)), rng.random((50, 3))])
    d = tess.Diagram(ctx, pts, LO, HI, vertex_capacity=capacity)
    got = d.cells_at_particles(sites)
    ref = orc.compute_at_points(pts, sites, LO, HI)
    for f in ("face_count", "face_offset", "neighbor"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    assert np.allclose(got["area"], ref["area"], rtol=1e-12, atol=0)
    d.close()
