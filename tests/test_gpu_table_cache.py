"""Shell tables of a program whose points move: a context does not keep one for
every grid shape it ever had, and a shape that comes back gets its table again."""
import ctypes as C

import numpy as np
import pytest

import tess

pytestmark = pytest.mark.gpu

LO, HI = np.full(3, -1.0), np.full(3, 2.0)


def _free(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


# tables of all 25^3 offsets, 187 KB each: 560 MB of them
def test_tables_do_not_pile_up():
    hip = tess._hip()
    base = tess.uniform(100, 4)
    with tess.Context(0) as c:
        first = tess.Diagram(c, base, LO, HI, density=0.05)
        first.compute()
        assert first.grid()[2] == 13
        want = first.cells()
        before = _free(hip)
        for k in range(3000):
            d = tess.Diagram(c, base * (1.0 + 1e-4 * (k + 1)), LO, HI, density=0.05)
            d.compute()
            d.close()
        assert before - _free(hip) < 320 << 20
        first.compute()
        got = first.cells()
        for f in want:
            assert np.array_equal(got[f], want[f]), f
        first.close()
