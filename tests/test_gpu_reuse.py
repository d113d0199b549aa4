"""Device blocks reused between objects: results do not depend on what a block
held before, on the size of the object it came from, or on which thread's
context freed it."""
import threading

import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)
FIELDS = ("volume", "face_count", "face_offset", "neighbor", "area")


def _cells(ctx, pts):
    d = tess.Diagram(ctx, pts, LO, HI)
    d.compute()
    out = d.cells()
    d.close()
    return out


# a block is handed out again for 8/9 of its size and more: equal, just inside,
# just outside and growing sizes
@pytest.mark.parametrize("sizes", [(9000, 9000), (9000, 8001, 9000), (9000, 7990, 12000)])
def test_diagrams_in_turn_and_from_threads(sizes):
    pts = [tess.uniform(n, 40 + k) for k, n in enumerate(sizes)]
    ref = [orc.compute(p, LO, HI) for p in pts]
    bad = []

    def work(first):
        with tess.Context(0) as c:
            for k in range(2 * len(sizes)):
                j = (first + k) % len(sizes)
                got = _cells(c, pts[j])
                for f in FIELDS:
                    same = np.array_equal(got[f], ref[j][f]) if f in ("face_count", "face_offset", "neighbor") \
                        else np.allclose(got[f], ref[j][f], rtol=1e-12, atol=0)
                    if not same:
                        bad.append((first, k, f))

    work(0)
    threads = [threading.Thread(target=work, args=(t,)) for t in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
