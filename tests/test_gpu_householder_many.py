"""M-orthonormalisation of many vectors: block sizes at the edges of the output
kernel's tiles of eight, of the coefficients' 48 vectors in LDS and of the 16
columns a workgroup beyond, up to every unit vector of the grid; checks and
tolerances of the smaller blocks.  And its time, which three kernels shared among
too few workgroups used to set at hundreds of vectors."""
import ctypes as C
import time

import numpy as np
import pytest

import test_gpu_products as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,k", [(16, 16, 7), (16, 16, 8), (16, 16, 48), (16, 16, 64), (16, 16, 65), (12, 18, 100),
                                     (16, 16, 128), (3, 4, 6)])
def test_orthonormalize_many(nx, ny, k):
    P.test_orthonormalize_edges(nx, ny, k, None)


def test_time_of_300_vectors():
    import maxwell_amd as M
    n, k = 64, 300
    rng = np.random.default_rng(0)
    G = M.Grid(np.ones((n, n)), 0.7, -1.3)
    v = [M.Edge(G, rng.standard_normal(2 * n * n) + 1j * rng.standard_normal(2 * n * n)) for _ in range(4)]
    x = [M.Edge(G) for _ in range(k)]
    best = 1.0
    for _ in range(4):
        for i in range(k):
            M.lib.copy_edge2d(v[i % 4].h, x[i].h)
        t = time.perf_counter()
        M.lib.orthonormalize_edge2d(k, (C.c_void_p * k)(*[e.h for e in x]), (M.Cplx * k)(), None)
        best = min(best, time.perf_counter() - t)
    print("300 vectors of 64 x 64: %.1f ms" % (1e3 * best))
    # a launch per product, update and fix, 300 times both ways, takes 18 ms
    assert best < 15e-3
