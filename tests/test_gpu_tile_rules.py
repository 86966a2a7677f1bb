"""mxh_afw_tile at the edges of the rules that choose between small tiles, whole
grids in LDS and square tiles, and with mode 16 (copies with their owner's
value) where the rules choose otherwise; checks and tolerances of the small
launches' comparison with the oracle.  Each choice has to be the faster form:
a grid is compared with one of the same tiles on the other side of the rule."""
import ctypes as C
import time

import numpy as np
import pytest

import test_gpu_few_vectors as F
from gpu_abi import NONE, Bloch, Dev, Level, vecs
from test_gpu_few_vectors import lib  # noqa: F401

pytestmark = pytest.mark.gpu


# 64 x 64 in FP64: 252 and 261 square tiles; 56 x 54 and 56 x 56: 3024 and 3136 nodes
@pytest.mark.parametrize("nx,ny,nv", [(64, 64, 28), (64, 64, 29), (56, 54, 26), (56, 56, 26)])
@pytest.mark.parametrize("mode,nsweep", [(1, 2), (5, 2), (8, 2), (10, 1)])
def test_whole_grids_and_square_tiles(lib, nx, ny, nv, mode, nsweep):  # noqa: F811
    F.test_small_launches(lib, 0, nx, ny, nv, False, mode, nsweep)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny,nv", [(12, 40, 3), (64, 64, 20), (62, 68, 20), (150, 162, 4), (290, 288, 1)])
@pytest.mark.parametrize("mode,nsweep", [(0, 1), (5, 2), (8, 2), (10, 1)])
def test_copies_with_their_owners_value(lib, prec, nx, ny, nv, mode, nsweep):  # noqa: F811
    F.test_small_launches(lib, prec, nx, ny, nv, False, mode | 16, nsweep)


def test_modes_that_do_not_exist_are_refused(lib):  # noqa: F811
    d = Dev(lib, np.zeros(2 * 2 * 64 * 64, complex))
    e = Dev(lib, np.zeros(2 * 2 * 64 * 64, complex))
    lv, bl = Level(64, 64, 1 / 64, 1 / 64), Bloch(1, 0, 1, 0, None, 1, None)
    for mode in (3, 9, 16 + 9, 32, 64):
        assert lib.mxh_afw_tile(0, C.byref(lv), C.byref(bl), 1, vecs(d, 8192), vecs(d, 8192), vecs(e, 8192), d.p, 1, mode,
                                NONE, NONE, NONE) != 0


def best_time(lib, nx, ny, nv, mode):  # noqa: F811
    N = nx * ny
    rng = np.random.default_rng(1)
    b = Dev(lib, rng.standard_normal((nv, 2 * N)) + 1j * rng.standard_normal((nv, 2 * N)))
    x, xo = Dev(lib, np.zeros((nv, 2 * N), complex)), Dev(lib, np.zeros((nv, 2 * N), complex))
    bc, xc = Dev(lib, np.zeros((nv, N // 2), complex)), Dev(lib, np.zeros((nv, N // 2), complex))
    eta = Dev(lib, np.ones(N))
    lv, bl = Level(nx, ny, 1 / 16, 1 / 16), Bloch(np.cos(1), np.sin(1), 1, 0, None, 1, None)
    best = 1.0
    for _ in range(20):
        t = time.perf_counter()
        for _ in range(20):
            assert lib.mxh_afw_tile(0, C.byref(lv), C.byref(bl), nv, vecs(b, 2 * N), vecs(x, 2 * N), vecs(xo, 2 * N),
                                    eta.p, 2, mode, NONE, vecs(bc, N // 2), vecs(xc, N // 2)) == 0
        assert lib.mxh_sync() == 0
        best = min(best, (time.perf_counter() - t) / 20)
    print("%d x %d, %d vectors, mode %d: %.1f us" % (nx, ny, nv, mode, 1e6 * best))
    return best


def test_time_of_few_vectors_on_the_largest_whole_grid(lib):  # noqa: F811
    assert best_time(lib, 64, 64, 16, 8) <= 1.15 * best_time(lib, 62, 68, 16, 8)


def test_time_of_one_vector_on_a_large_grid(lib):  # noqa: F811
    assert best_time(lib, 384, 384, 1, 8) <= 0.95 * best_time(lib, 384, 384, 1, 24)
