"""Downloads that the staging is not the way for: one small array, pinned
destinations, and small results while another thread's large ones come down."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import tess

pytestmark = pytest.mark.gpu

LO, HI = np.zeros(3), np.ones(3)
FIELDS = ("volume", "face_count", "face_offset", "neighbor", "area")


class Pinned:
    def __init__(self, like):
        self.hip, self.p, self.like = tess._hip(), C.c_void_p(), like
        assert self.hip.hipHostMalloc(C.byref(self.p), C.c_size_t(like.nbytes + 16), 0) == 0
        self.bytes = np.ctypeslib.as_array(C.cast(self.p, C.POINTER(C.c_uint8)), (like.nbytes + 16,))
        self.bytes[:] = 0xA5

    def check(self):
        assert np.array_equal(self.bytes[: self.like.nbytes].view(self.like.dtype), self.like)
        assert (self.bytes[self.like.nbytes:] == 0xA5).all()  # nothing past the array's end

    def close(self):
        self.hip.hipHostFree(self.p)


def _ms(f, reps):
    t = []
    for _ in range(reps):
        a = time.perf_counter()
        f()
        t.append(time.perf_counter() - a)
    return 1e3 * sorted(t)[reps // 2]


# one to five arrays on both sides of 64 KiB (k - 1)^2, some NULL, and pinned
# beside pageable ones
@pytest.mark.parametrize("n", [1, 3, 700, 3001, 6007, 130001])
def test_pinned_destinations(ctx, n):
    d = tess.Diagram(ctx, tess.uniform(n, n), LO, HI)
    d.compute()
    got = d.cells()
    for which in ("0", "2", "4", "01", "34", "024", "0123", "01234"):
        for mixed in (False, True):
            args, pins, plain = [None] * 5, [], []
            for k in map(int, which):
                if mixed and k == int(which[-1]):
                    plain.append((k, np.zeros_like(got[FIELDS[k]])))
                    args[k] = C.c_void_p(plain[-1][1].ctypes.data)
                else:
                    pins.append(Pinned(got[FIELDS[k]]))
                    args[k] = pins[-1].p
            ctx.check(ctx.lib.tess_diagram_copy_cells(d.h, *args))
            for p in pins:
                p.check()
                p.close()
            for k, a in plain:
                assert np.array_equal(a, got[FIELDS[k]])
    d.close()


# the offsets of a set of a batch count from its own first face
def test_pinned_destinations_of_a_batch(ctx):
    b = tess.Batch(ctx, [(tess.uniform(n, n), LO, HI) for n in (500, 4000, 40000)])
    b.compute()
    for k in range(3):
        got = b.cells(k)
        for which in ("2", "01234"):
            pins = {int(j): Pinned(got[FIELDS[int(j)]]) for j in which}
            ctx.check(ctx.lib.tess_batch_copy_cells(b.h, k, *[pins[j].p if j in pins else None for j in range(5)]))
            for p in pins.values():
                p.check()
                p.close()
    b.close()


# to pinned memory the call costs what the runtime's own copy does (twice that
# by way of the staging)
def test_pinned_download_time(ctx):
    d = tess.Diagram(ctx, tess.uniform(120000, 2), LO, HI)
    d.compute()
    area = d.cells()["area"]
    pin, src = Pinned(area), tess.DeviceArray(ctx, area)
    args = [None, None, None, None, pin.p]
    hip = tess._hip()
    for f in (lambda: hip.hipMemcpy(pin.p, src.ptr, area.nbytes, 2), lambda: ctx.lib.tess_diagram_copy_cells(d.h, *args)):
        _ms(f, 5)
    raw = _ms(lambda: hip.hipMemcpy(pin.p, src.ptr, area.nbytes, 2), 31)
    call = _ms(lambda: ctx.lib.tess_diagram_copy_cells(d.h, *args), 31)
    pin.check()
    pin.close()
    d.close()
    assert call < 1.6 * raw, (call, raw)


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
