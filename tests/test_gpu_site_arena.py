"""Cells of outside sites with more faces together than the call's arena holds
(64 a site, 2^16 at least): refused, as the diagram's own cells are, not
returned without faces."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)


def test_full_arena(ctx):
    rng = np.random.default_rng(7)
    pts = rng.random((1500, 3)) * [1, 1e-4, 1]  # a sheet: a site off it has a face with nearly every point
    sites = np.c_[rng.random(60), rng.uniform(0.3, 0.9, 60), rng.random(60)]
    d = tess.Diagram(ctx, pts, LO, HI)
    few = d.cells_at_particles(sites[:3])
    ref = orc.compute_at_points(pts, sites, LO, HI)
    assert np.array_equal(few["face_count"], ref["face_count"][:3])
    assert np.allclose(few["volume"], ref["volume"][:3], rtol=1e-9, atol=0)
    assert ref["face_count"].sum() > 1 << 16
    with pytest.raises(tess.TessError, match="TESS_E_CAPACITY"):
        d.cells_at_particles(sites)
    again = d.cells_at_particles(sites[:3])  # the next call has the whole arena
    assert np.array_equal(again["neighbor"], few["neighbor"])
    d.close()
