"""Results written to the host by one kernel: arrays of odd lengths and odd
alignment side by side, in one chunk and in several, and single cells from the
smallest capacity up."""
import ctypes as C

import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)
FIELDS = ("volume", "face_count", "face_offset", "neighbor", "area")


# 1 MiB (one chunk) lies between 5,000 and 5,200 cells; 20,011 take four chunks
@pytest.mark.parametrize("n", [1, 2, 3, 5, 5000, 5200, 20011])
def test_arrays_together_and_one_by_one(ctx, n):
    pts = tess.uniform(n, n)
    d = tess.Diagram(ctx, pts, LO, HI)
    d.compute()
    got = d.cells()
    ref = orc.compute(pts, LO, HI)
    for f in ("face_count", "face_offset", "neighbor"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    assert np.allclose(got["area"], ref["area"], rtol=1e-12, atol=0)
    for k, f in enumerate(FIELDS):
        alone = np.zeros_like(got[f])
        args = [None] * 5
        args[k] = C.c_void_p(alone.ctypes.data)
        ctx.check(ctx.lib.tess_diagram_copy_cells(d.h, *args))
        assert np.array_equal(alone, got[f]), f
    d.close()


# every set starts at the next point: all alignments of 4- and 8-byte arrays
@pytest.mark.parametrize("sizes", [(1, 1, 2, 3, 5, 64, 63, 65, 1), (1001, 7, 5300, 2, 999)])
def test_sets_of_a_batch(ctx, sizes):
    sets = [(tess.uniform(n, 7 + k), LO, HI) for k, n in enumerate(sizes)]
    b = tess.Batch(ctx, sets)
    b.compute()
    for k, (pts, _, _) in enumerate(sets):
        d = tess.Diagram(ctx, pts, LO, HI)
        d.compute()
        one, of_batch = d.cells(), b.cells(k)
        for f in FIELDS:
            assert np.array_equal(one[f], of_batch[f]), (k, f)
        d.close()
    b.close()


# points on a sphere of radius 0.45 and its centre: the centre's cell has
# about 2 (n - 2) vertices
@pytest.mark.parametrize("n", [20, 30, 33, 34, 36, 60, 64, 68, 100])
def test_single_cells_by_capacity(ctx, n):
    rng = np.random.default_rng(n)
    p = rng.normal(size=(n, 3))
    pts = np.vstack([p / np.linalg.norm(p, axis=1)[:, None] * 0.45 + 0.5, [[0.5, 0.5, 0.5]]])
    d = tess.Diagram(ctx, pts, LO, HI)
    ref = orc.compute_geometry(pts, LO, HI)
    fo = ref["face_offset"].astype(int)
    for i in (0, n // 2, n):
        if ref["face_count"][i] > 64:  # more faces than a single cell may have
            with pytest.raises(tess.TessError, match="TESS_E_CAPACITY"):
                d.get_cell_at_index(i)
            continue
        c = d.get_cell_at_index(i)
        s = slice(fo[i], fo[i + 1])
        assert np.array_equal(c.compute_neighbors(), ref["neighbor"][s])
        assert c.compute_volume() == pytest.approx(ref["volume"][i], rel=1e-12)
        areas = np.array([c.face(f)[0] for f in range(c.face_count())])
        assert np.allclose(areas, ref["area"][s], rtol=1e-12, atol=0)
        ro = ref["ring_offset"].astype(int)
        assert [len(c.face_vertices(f)) for f in range(c.face_count())] == \
            [ro[f + 1] - ro[f] for f in range(fo[i], fo[i + 1])]
        rings = np.unique(np.concatenate([c.face_vertices(f) for f in range(c.face_count())]), axis=0)
        assert np.array_equal(rings, np.unique(c.compute_vertices(), axis=0))
    d.close()
