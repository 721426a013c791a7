"""nbx_simp_filter waits for no other handle's work: it returns while another
stream of the kind the handles have (one the legacy stream waits for) still holds
a host function back.  And it still answers after the system it was made from is
gone."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_filter_waits_for_no_other_stream():
    from nbots_amd import load, synth
    from nbots_amd.fem import Fem, Simp
    hip = load()   # (symbols are looked up in what the library is linked with, too)
    f = Fem.from_problem(synth.cantilever_point(32, 16, jitter=0.1))
    s = Simp(f, rmin=1.5)
    want = s.filter()
    go, held = threading.Event(), threading.Event()

    @C.CFUNCTYPE(None, C.c_void_p)
    def hold(_):
        held.set()
        go.wait(3.0)   # (ends by itself: no call can hang on it)

    stream = C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    assert hip.hipLaunchHostFunc(stream, hold, None) == 0
    assert held.wait(10.0)
    t = time.perf_counter()
    got = s.filter()
    waited = time.perf_counter() - t
    go.set()
    assert hip.hipStreamSynchronize(stream) == 0
    assert hip.hipStreamDestroy(stream) == 0
    print(waited)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)
    assert waited < 1.0
    f.destroy()
    for a, b in zip(s.filter(), want):
        assert np.array_equal(a, b)
    s.destroy()
