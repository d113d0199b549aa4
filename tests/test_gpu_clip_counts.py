"""Counters of the 64-vertex clip on nearly degenerate points, where cuts take
its slot, general and capacity routes, against the 128-vertex kernel's, whose
clip is another one."""
import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sigma", [0.0, 1e-12, 1e-9, 1e-6, 1e-3])
@pytest.mark.parametrize("cells", [5, 8])
def test_counts_on_jittered_lattices(ctx, sigma, cells):
    pts = tess.fcc(11, cells, 1.0, sigma)
    lo, hi = np.minimum(pts.min(0), 0) - 1e-9, np.maximum(pts.max(0), cells) + 1e-9
    got, answers = [], []
    for capacity in (64, 128):
        d = tess.Diagram(ctx, pts, lo, hi, density=5.0, vertex_capacity=capacity, collect_stats=True)
        answers.append(d.compute_status())  # (1e-12 is the clip's tolerance: cells that fail their checks)
        s = d.stats()
        # cells past 64 vertices are counted by the pass that finished them
        got.append({f: s[f] for f in ("flops", "classified", "cuts", "entries", "incident_cuts", "max_vertices", "r2", "status")})
        d.close()
    assert answers[0] == answers[1]
    for f in got[0]:
        assert np.array_equal(got[0][f], got[1][f]), f
    if answers[0] != tess.TESS_OK:
        return
    ref = orc.compute(pts, lo, hi, density=5.0)["stats"]
    for f in ("classified", "cuts", "incident_cuts"):
        assert np.array_equal(got[0][f], ref[f]), f
