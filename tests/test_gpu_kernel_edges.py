"""The cut, query and network kernels at the edges of their tiles and routes,
against the oracle (exact where the results are), and the network against
itself (a row's output does not depend on the rows beside it)."""
import numpy as np
import pytest

import tess
from oracle import mlp
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

COUNTERS = ("streamed", "classified", "cuts", "entries", "flops", "incident_cuts")


def _lattice(k):
    return np.stack(np.meshgrid(*[(np.arange(k) + 0.5) / k] * 3, indexing="ij"), -1).reshape(-1, 3)


def _sphere(n):
    p = np.random.default_rng(n).normal(size=(n, 3))
    return np.vstack([p / np.linalg.norm(p, axis=1)[:, None] * 0.45 + 0.5, [[0.5, 0.5, 0.5]]])


# vertices on the cutting plane (lattices); more than 64 pairs, hence the
# second pair register and crossings in it (centres of spheres, 3 (n - 2)
# pairs); more than 64, 128 and 256 vertices (reruns and the spill kernel);
# dead slots below the highest live one (random sets)
CLIP_SETS = {
    "lattice 5": lambda: _lattice(5),
    "lattice 9": lambda: _lattice(9),
    "fcc": lambda: tess.fcc(7, 6, 1.0, 0.0) / 6.0,
    "fcc jittered": lambda: tess.fcc(7, 6, 1.0, 1e-9) / 6.001 + 1e-5,
    "sphere 24": lambda: _sphere(24),
    "sphere 34": lambda: _sphere(34),
    "sphere 60": lambda: _sphere(60),
    "sphere 140": lambda: _sphere(140),
    "uniform": lambda: tess.uniform(3000, 1),
    "clustered": lambda: tess.clustered(3000, 2),
    "two planes": lambda: np.concatenate([tess.uniform(300, 3) * [1, 1, 0] + [0, 0, z] for z in (0.25, 0.75)]),
}


@pytest.mark.parametrize("density", [1.25, 5.0])
@pytest.mark.parametrize("name", CLIP_SETS)
def test_cells_and_counters(ctx, name, density):
    pts = CLIP_SETS[name]()
    lo, hi = np.zeros(3), np.ones(3)
    d = tess.Diagram(ctx, pts, lo, hi, density=density, collect_stats=True)
    d.compute()
    got, st = d.cells(), d.stats()
    ref = orc.compute(pts, lo, hi, density=density)
    for f in ("face_count", "face_offset", "neighbor"):
        assert np.array_equal(got[f], ref[f]), f
    assert np.allclose(got["volume"], ref["volume"], rtol=1e-12, atol=0)
    assert np.allclose(got["area"], ref["area"], rtol=1e-12, atol=0)
    for f in COUNTERS:
        # vertices 1e-9 apart: in a few cells the oracle's walk keeps another
        # number of them for some cuts, and counts other operations, while
        # every face, area and count of cuts is the same
        if f == "flops" and name == "fcc jittered":
            continue
        assert np.array_equal(st[f].astype(np.float64), ref["stats"][f].astype(np.float64)), f
    t = d.timings()
    if not (t["capacity_reruns"] or t["table_reruns"] or t["spill_cells"]):
        # every cell counted once: the summary's slots add up to the cells' own
        assert t["flops"] == int(st["flops"].sum())
        assert t["incident_cuts"] == int(st["incident_cuts"].sum())
    d.close()


def _dense(n_run):
    """Grid cells of n_run points beside empty ones and single points."""
    rng = np.random.default_rng(n_run)
    spots = rng.random((12, 3))
    pts = np.concatenate([s + 1e-4 * rng.random((n_run, 3)) for s in spots] + [rng.random((200, 3))])
    return np.clip(pts, 0.0, 1.0)


# 16 queries a workgroup's wavefronts take four at a time; rows of a box above
# 16 (a query's lanes) at the largest radius; rows of 48 points and more are
# walked by the whole wavefront
@pytest.mark.parametrize("nq", [1, 3, 4, 15, 16, 17, 65])
@pytest.mark.parametrize("points", ["uniform", "flat", "runs 3", "runs 47", "runs 48", "runs 65", "runs 200"])
def test_queries(ctx, nq, points):
    rng = np.random.default_rng(nq)
    if points.startswith("runs"):
        pts = _dense(int(points.split()[1]))
    else:
        pts = rng.random((4000, 3))
        if points == "flat":
            pts[:, 1] = 0.5
    groups = (np.arange(len(pts)) % 3).astype(np.int64)
    q = np.concatenate([pts[rng.integers(0, len(pts), nq)][: nq // 2], rng.random((nq - nq // 2, 3)) * 1.4 - 0.2])
    radii = rng.choice([0.0, -1.0, np.nan, np.inf, 1e-300, 0.02, 0.1, 0.3, 0.7, 2.0], nq)
    d = tess.Diagram(ctx, pts, np.full(3, -0.5), np.full(3, 1.5), density=2.0, groups=groups)
    d.compute()
    for kind in (tess.QUERY_CELLS, tess.QUERY_CELL_RADIUS, tess.QUERY_REAL_RADIUS, tess.QUERY_CLOUD):
        for r in (radii, 0.15):
            off, ids = d.query(kind, q, r)[:2]
            ro, ri = orc.queries(kind, pts, q, r, density=2.0)
            assert np.array_equal(off, ro) and np.array_equal(ids, ri), (kind, np.ndim(r))
    off, ids = d.query(tess.QUERY_CLOUD, q, radii, target_group=1)[:2]
    ro, ri = orc.queries(tess.QUERY_CLOUD, pts, q, radii, density=2.0, groups=groups, target_group=1)
    assert np.array_equal(off, ro) and np.array_equal(ids, ri)
    d.close()


# enough queries to be taken in grid order, at an odd count
@pytest.mark.parametrize("points", ["uniform", "runs 48"])
def test_queries_in_grid_order(ctx, points):
    rng = np.random.default_rng(5)
    pts = _dense(48) if points.startswith("runs") else rng.random((20000, 3))
    q = rng.random((33333, 3)) * 1.2 - 0.1
    d = tess.Diagram(ctx, pts, np.full(3, -0.5), np.full(3, 1.5), density=2.0)
    d.compute()
    for kind in (tess.QUERY_CELLS, tess.QUERY_CELL_RADIUS, tess.QUERY_REAL_RADIUS, tess.QUERY_CLOUD):
        off, ids = d.query(kind, q, 0.03)[:2]
        ro, ri = orc.queries(kind, pts, q, 0.03, density=2.0)
        assert np.array_equal(off, ro) and np.array_equal(ids, ri), kind
    d.close()


def _samples(n, seed):
    rng = np.random.default_rng(seed)
    x = np.zeros((n, mlp.IN), np.float32)
    x[:, :mlp.FEATURES] = np.log1p(rng.poisson(rng.uniform(1, 60, (n, 1)), (n, mlp.FEATURES)))
    return mlp.bf16_bits(x), rng.normal(0, 1, (n, 2)).astype(np.float32)


# tiles of 16 rows, 64 per workgroup, and more rows than all workgroups hold
def test_forward_rows_are_independent(ctx):
    m = tess.Model(ctx, seed=3)
    x, _ = _samples(70001, 4)
    y = m.forward(x)
    for n in (1, 15, 16, 17, 63, 64, 65, 1023, 65535, 65537):
        assert np.array_equal(m.forward(x[:n]), y[:n]), n
    m.close()


# one sample, the last of 32 and one more; 1, 2 and 63 to 65 slots of 32, 255
# to 257: the slots are added up 4 wavefronts at a time.  The bound is the one
# of the gradient test beside the learned search: bf16 activations against the
# reference's rounding.
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 32 * 63, 32 * 64, 32 * 64 + 1, 32 * 255 + 7, 32 * 256, 32 * 257])
def test_gradient_slots(ctx, n):
    m = tess.Model(ctx, seed=5)
    p = mlp.init_params(5)
    m.set(p)
    x, t = _samples(n, 6 + n)
    loss, g = m.gradient(x, t)
    ref_loss, ref = mlp.gradient(p, x, t, rounded=True)
    assert loss == pytest.approx(ref_loss, rel=1e-3)
    assert np.linalg.norm(g - ref) < 5e-3 * np.linalg.norm(ref)
    m.close()


# grids of one, two and three cells per dimension: every neighbourhood of 27
# cells is cut off at the walls
@pytest.mark.parametrize("n,density", [(1, 5.0), (30, 5.0), (100, 5.0), (1000, 1.25)])
def test_features_and_predictions(ctx, n, density):
    pts = tess.uniform(n, 11)
    d = tess.Diagram(ctx, pts, np.zeros(3), np.ones(3), density=density, collect_stats=True)
    d.compute()
    cell, _, delim = d.copy_grid()
    cpd = d.grid()[2]
    feat = d.features()
    assert np.array_equal(feat, mlp.features(cell, delim, cpd))
    m = tess.Model(ctx, seed=2)
    m.set(mlp.init_params(2), norm=np.array([0.1, 0.7, 4.0, 0.5], np.float32),
          calib=np.array([np.inf, np.inf, 0, 0], np.float32))
    y = m.forward(feat).astype(np.float64)
    out = d.predict(m)
    smin = d.grid()[1].min()
    want = np.stack([np.exp(np.float32(0.7) * y[:, 0] + np.float32(0.1)) * smin,
                     np.expm1(np.float32(0.5) * y[:, 1] + np.float32(4.0))], 1)
    # a value computed in double, then rounded to float
    assert np.allclose(out, want, rtol=2.0**-22, atol=0)
    m.close()
    d.close()


# the largest radius decides how long a shell table the clouds need: negative
# ones alone, none, one past the default table, infinite and NaN ones, at the
# first, a middle and the last place of one and of several workgroups' radii
@pytest.mark.parametrize("nq", [2, 255, 1025, 5000])
@pytest.mark.parametrize("odd", [None, 0.9, np.inf, np.nan, -np.inf])
def test_cloud_radii_on_the_device(ctx, nq, odd):
    rng = np.random.default_rng(nq)
    pts, q = rng.random((6000, 3)), rng.random((nq, 3))
    d = tess.Diagram(ctx, pts, np.zeros(3), np.ones(3), density=1.25)
    d.compute()
    for base in (0.01, -1.0):
        for at in (0, nq // 2, nq - 1):
            r = np.full(nq, base)
            if odd is not None:
                r[at] = odd
            qt, rt = tess.DeviceArray(ctx, q), tess.DeviceArray(ctx, r)
            res = d.query_device(tess.QUERY_CLOUD, qt.ptr, nq, rt.ptr, nq)
            off, ids = res.copy()
            ro, ri = orc.queries(tess.QUERY_CLOUD, pts, q, r, density=1.25)
            assert np.array_equal(off, ro) and np.array_equal(ids, ri), (base, at)
            res.close()
    d.close()


# clouds are counted by 16 lanes each from 16,384 queries on; radii from none
# to the whole table's, mixed within a wavefront
@pytest.mark.parametrize("nq", [16383, 16384, 16385, 20001])
@pytest.mark.parametrize("grouped", [False, True])
def test_many_clouds(ctx, nq, grouped):
    rng = np.random.default_rng(nq)
    pts, q = rng.random((3000, 3)), rng.random((nq, 3)) * 1.2 - 0.1
    groups = (np.arange(len(pts)) % 3).astype(np.int64)
    r = rng.choice([-1.0, 0.0, 1e-300, 0.005, 0.01, 0.02], nq)
    r[:: nq // 7] = 0.6
    d = tess.Diagram(ctx, pts, np.full(3, -0.5), np.full(3, 1.5), density=1.25, groups=groups)
    d.compute()
    off, ids = d.query(tess.QUERY_CLOUD, q, r, target_group=1 if grouped else None)[:2]
    ro, ri = orc.queries(tess.QUERY_CLOUD, pts, q, r, density=1.25, groups=groups, target_group=1 if grouped else -1)
    assert np.array_equal(off, ro) and np.array_equal(ids, ri)
    d.close()
