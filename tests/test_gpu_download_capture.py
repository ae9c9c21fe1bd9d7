"""A field download while a stream of the program is being captured.

With a capture in global mode open, HIP refuses waits to threads in that mode
and leaves them to threads in relaxed mode.  A download keeps to the mode of the
thread that calls it, with whatever threads it moves the chunks on.
"""
import ctypes as C

import numpy as np
import pytest

from tam_amd import configs, lib

pytestmark = pytest.mark.gpu

GLOBAL, THREAD_LOCAL, RELAXED = range(3)


def _hip():
    lib.load()
    return C.CDLL("libamdhip64.so")


# results of one, two and more slots of 2 MiB: one thread, two, eight
@pytest.mark.parametrize("n", [40, 64, 82, 130])
@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL, RELAXED])
def test_a_relaxed_thread_downloads_during_a_capture(n, mode):
    print("case", n, mode, flush=True)
    g = configs.three_layer_skin(n=(n, n, n), ext=(2.0, 2.0, 1.0), packets=1, steps=1).grid()
    g.mc_run(20_000, seed=1)
    want = [g.download(f) for f in (lib.FIELD_TALLY, lib.FIELD_TEMP, lib.FIELD_MAT)]
    hip = _hip()
    s, graph, m = C.c_void_p(), C.c_void_p(), C.c_int(RELAXED)
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    assert hip.hipThreadExchangeStreamCaptureMode(C.byref(m)) == 0            # m: the thread's own
    try:
        assert hip.hipStreamBeginCapture(s, mode) == 0
        try:
            got = [g.download(f) for f in (lib.FIELD_TALLY, lib.FIELD_TEMP, lib.FIELD_MAT)]
        finally:
            rc = hip.hipStreamEndCapture(s, C.byref(graph))
    finally:
        hip.hipThreadExchangeStreamCaptureMode(C.byref(m))
    assert rc == 0                                                            # and the capture is whole
    for a, b in zip(want, got):
        assert np.array_equal(a, b)
    hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(s)
    g.close()


@pytest.mark.parametrize("n", [64, 130])
def test_a_refused_download_leaves_the_ring_sound(n):
    """In global mode the wait is refused, as it is without the ring; the
    copies that were sent end before another download has their slots."""
    print("case", n, flush=True)
    a, b = (configs.three_layer_skin(n=(n, n, n), ext=(2.0, 2.0, 1.0), packets=1, steps=1).grid() for _ in range(2))
    for q, g in enumerate((a, b)):
        g.upload(lib.FIELD_JMEAN, np.random.default_rng(q).random((n, n, n)))
    want = b.download(lib.FIELD_JMEAN)
    hip = _hip()
    s, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    assert hip.hipStreamBeginCapture(s, GLOBAL) == 0
    try:
        with pytest.raises(lib.TamError):
            a.download(lib.FIELD_JMEAN)
    finally:
        hip.hipStreamEndCapture(s, C.byref(graph))                            # the refusal has ended it
    hip.hipGetLastError()
    for _ in range(3):
        assert np.array_equal(b.download(lib.FIELD_JMEAN), want)
    assert np.array_equal(a.download(lib.FIELD_JMEAN), np.random.default_rng(0).random((n, n, n)))
    hip.hipStreamDestroy(s)
    a.close()
    b.close()
