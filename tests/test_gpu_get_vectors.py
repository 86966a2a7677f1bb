"""mx_get_vectors hands a problem's vectors over at the price of one copy: on small
grids (dense blocks) against a plain copy of the same bytes; and it hands over
the right ones on both sides of the size from which blocks are padded."""
import ctypes as C
import time

import numpy as np
import pytest

import oracle as O
from gpu_abi import Dev, bind

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,levels,method", [(64, 4, 0), (128, 5, 1), (256, 6, 0), (256, 6, 1)])
def test_vectors_are_the_ritz_vectors(n, levels, method):
    import maxwell_amd as M
    eta, k = O.rod_eta(n), [(0.4, -1.1), (2.0, 0.3)]
    S = M.Solver(eta, n0=4, levels=levels, block=4, max_problems=2, method=method)
    r = S.solve([a for a, _ in k], [b for _, b in k], neig=2, tol=1e-8, maxit=200, seed=3)
    assert r["converged"].all()
    for p, (kx, ky) in enumerate(k):
        g = O.Grid2D(eta, kx=kx, ky=ky)
        for i, e in enumerate(S.vectors(p)[:2]):
            lam, Me = r["lam"][p, i], O.addeval(g, 0.0, 1.0, e)
            res = O.addeval(g, 1.0, 0.0, e) - lam * Me
            # the residual the solve stopped at, and its own rounding
            assert np.linalg.norm(res) <= 2e-8 * lam * np.linalg.norm(Me)
    S.close()


def test_time_on_a_small_grid():
    import maxwell_amd as M
    L = bind(M.lib)
    S = M.Solver(O.rod_eta(64), n0=4, levels=4, block=12, max_problems=2)
    S.solve([0.4, 1.0], [0.2, 0.1], neig=10, maxit=1)
    out = np.zeros(12 * S.nedge, np.complex128)
    d = Dev(L, None, nbytes=out.nbytes)
    ptr = out.view(np.float64).ctypes.data_as(C.POINTER(C.c_double))

    def best(f):
        t = []
        for _ in range(60):
            t0 = time.perf_counter()
            assert f() == 0
            t.append(time.perf_counter() - t0)
        return min(t)

    get = best(lambda: M.lib.mx_get_vectors(S.h, 1, ptr))
    copy = best(lambda: L.mxh_d2h(out.ctypes.data_as(C.c_void_p), d.p, out.nbytes))
    S.close()
    print("vectors %.0f us, a copy of their bytes %.0f us" % (1e6 * get, 1e6 * copy))
    assert get <= 1.25 * copy
