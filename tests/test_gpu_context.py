"""Contexts made while a stream of the process is being captured."""
import ctypes as C
import threading

import numpy as np
import pytest

import tess
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


# capture modes global, thread-local and relaxed; from the capturing thread
# and from another
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("other", [False, True])
def test_context_during_a_capture(ctx, mode, other):
    hip = tess._hip()
    stream, graph, made = C.c_void_p(), C.c_void_p(), []

    def make():
        try:
            made.append(tess.Context(0))
        except tess.TessError as e:
            made.append(e)

    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    if other:
        t = threading.Thread(target=make)
        t.start()
        t.join()
    else:
        make()
    hip.hipStreamEndCapture(stream, C.byref(graph))  # (may have been given up by the runtime)
    if graph:
        hip.hipGraphDestroy(graph)
    hip.hipGetLastError()
    assert hip.hipStreamDestroy(stream) == 0
    c, = made
    assert isinstance(c, tess.Context), c
    pts = tess.uniform(500, 3)
    d = tess.Diagram(c, pts, np.zeros(3), np.ones(3))
    d.compute()
    got, want = d.cells(), orc.compute(pts, np.zeros(3), np.ones(3))
    assert np.array_equal(got["neighbor"], want["neighbor"])
    assert np.allclose(got["volume"], want["volume"], rtol=1e-12, atol=0)
    d.close()
    c.close()
