"""mxh_coarse_inverse at the edges of its row blocks (64 rows a lane block, eight
steps a load, two columns a wave), and its time.

Tolerance: forward and back substitution with a Cholesky factor of condition
sqrt(cond A) leave an error of at most n eps cond(A) |A^-1|; the matrices have
a condition below 1e3.  What lies above the diagonal is not read."""
import ctypes as C
import time

import numpy as np
import pytest

from gpu_abi import Dev, bind

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    L = bind(M.lib)
    L.mxh_coarse_inverse.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    return L


def factors(n, nprob, rng):
    A, L = [], []
    for _ in range(nprob):
        q = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))[0]
        a = (q * np.geomspace(1.0, 500.0, n)) @ q.conj().T
        a = 0.5 * (a + a.conj().T)
        l = np.linalg.cholesky(a)
        l[np.triu_indices(n, 1)] = np.nan
        A.append(a)
        L.append(l.T)  # column-major
    return np.stack(A), np.ascontiguousarray(np.stack(L))


@pytest.mark.parametrize("n", [1, 2, 8, 9, 32, 63, 64, 65, 72, 127, 128, 129, 200, 255, 256])
def test_inverse(lib, n):
    print("coarse inverse of %d rows" % n, flush=True)
    P = 3
    A, L = factors(n, P, np.random.default_rng(n))
    dL, dW = Dev(lib, L), Dev(lib, np.zeros((P, n, n), complex))
    assert lib.mxh_coarse_inverse(n, P, dL.p, dW.p) == 0
    ref = np.linalg.inv(A)
    assert np.abs(dW.get() - ref).max() <= n * 2.2e-16 * 500.0 * np.abs(ref).max()


def test_sizes_outside_are_refused(lib):
    assert lib.mxh_coarse_inverse(0, 1, None, None) != 0
    assert lib.mxh_coarse_inverse(257, 1, None, None) != 0
    assert lib.mxh_coarse_inverse(32, 0, None, None) != 0


@pytest.mark.parametrize("n,P", [(72, 1), (200, 1), (200, 64)])
def test_time(lib, n, P):
    """A solve pays for the inverses of its coarse matrices before its first step,
    a cycle of the module API whenever its matrix changes: against the
    milliseconds of a short solve that has to stay below one."""
    _, L = factors(n, 1, np.random.default_rng(n))
    dL, dW = Dev(lib, np.repeat(L, P, 0)), Dev(lib, np.zeros((P, n, n), complex))
    best = 1.0
    for _ in range(10):
        t = time.perf_counter()
        for _ in range(3):
            assert lib.mxh_coarse_inverse(n, P, dL.p, dW.p) == 0
        assert lib.mxh_sync() == 0
        best = min(best, (time.perf_counter() - t) / 3)
    print("%d rows, %d problems: %.0f us" % (n, P, 1e6 * best))
    assert best < (0.3e-3 if n == 72 else 1e-3 if P == 1 else 3e-3)
