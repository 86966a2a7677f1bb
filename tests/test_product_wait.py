"""The wait for a product's mark (no GPU: the mark is a plain number in memory):
there or not, and how long it goes on where it does not come."""
import ctypes as C
import threading
import time

import numpy as np

import maxwell_amd as M


def wait(a, mark, us):
    f = M.lib.mxh_product_wait
    f.argtypes = [C.c_void_p, C.c_double, C.c_double]
    t = time.perf_counter()
    r = f(a.ctypes.data_as(C.c_void_p), mark, us)
    return r, 1e6 * (time.perf_counter() - t)


def test_mark_that_is_there():
    assert wait(np.array([0.0, 0.0, 7.0]), 7.0, 0.0)[0] == 1


def test_mark_that_comes():
    a = np.zeros(3)
    timer = threading.Timer(0.02, lambda: a.__setitem__(2, 3.0))
    timer.start()
    assert wait(a, 3.0, 5e6)[0] == 1
    timer.join()


def test_wait_ends_at_its_limit():
    a = np.zeros(3)
    for us in (0.0, 40.0, 1000.0):
        runs = [wait(a, 1.0, us) for _ in range(20)]
        assert all(r == 0 for r, _ in runs)
        # the limit, one turn of 32 looks beyond it, and the call (the least of 20 runs)
        assert us <= min(t for _, t in runs) <= us + 50.0
