"""Downloads that the staging is not the way for: small results while another
thread's large ones come down."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import tess

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)
FIELDS = ("volume", "face_count", "face_offset", "neighbor", "area")


def _ms(f, reps):
    t = []
    for _ in range(reps):
        a = time.perf_counter()
        f()
        t.append(time.perf_counter() - a)
    return 1e3 * sorted(t)[reps // 2]


# one thread brings down 240 MB again and again; a single cell on the same
# context does not wait until it has finished
def test_small_results_beside_large_ones(ctx):
    big = tess.Diagram(ctx, tess.uniform(1000000, 5), LO, HI, density=5.0)
    big.compute()
    small = tess.Diagram(ctx, tess.uniform(20000, 6), LO, HI)
    small.compute()
    want = small.get_cell_at_index(7).compute_volume()
    out = big.cells()
    again = {f: np.zeros_like(out[f]) for f in FIELDS}
    args = [C.c_void_p(again[f].ctypes.data) for f in FIELDS]
    alone = _ms(lambda: ctx.lib.tess_diagram_copy_cells(big.h, *args), 5)
    stop = threading.Event()

    def loop():
        while not stop.is_set():
            ctx.lib.tess_diagram_copy_cells(big.h, *args)

    t = threading.Thread(target=loop)
    t.start()
    try:
        time.sleep(0.05)
        ms = _ms(lambda: small.get_cell_at_index(7), 15)
        assert small.get_cell_at_index(7).compute_volume() == want
    finally:
        stop.set()
        t.join()
    for f in FIELDS:
        assert np.array_equal(again[f], out[f]), f
    big.close()
    small.close()
    assert ms < alone / 2, (ms, alone)
