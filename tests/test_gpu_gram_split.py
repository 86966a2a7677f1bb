"""Gram sums of blocks of more than three tiles (24 vectors) where few
workgroups run: the tiles after the third in workgroups of their own.  Values at
the edges of the tiles, with and without column lists, on grids and problem
counts on both sides of the choice, against the sums written out; and the time
of a small grid's wide block, which is that of one workgroup's chain."""
import ctypes as C
import time

import numpy as np
import pytest

from gpu_abi import Bloch, Dev, Level, bind, vecs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    return bind(M.lib)


def reference(u, eta):
    m, _, ny, nx = u.shape
    x, y = u[:, 0], u[:, 1]
    xu, yr = np.roll(x, -1, 1), np.roll(y, -1, 2)
    xu[:, -1] *= np.exp(-1.3j)
    yr[:, :, -1] *= np.exp(0.7j)
    c = (x - xu - y + yr).reshape(m, -1)
    mx, my = 0.08 / 0.1 / 6.0, 0.1 / 0.08 / 6.0
    f = lambda a, b: a.reshape(m, -1).conj() @ b.reshape(m, -1).T
    return (c.conj() @ (eta.ravel() * c).T,
            mx * (4 * f(x, x) + f(x, xu) + f(xu, x)) + my * (4 * f(y, y) + f(y, yr) + f(yr, y)))


# every form: few problems of small grids (split after the third tile), nine of 72 x
# 90 (after the fifth, whole up to five), many problems (whole); grids of fewer than
# four strips (16, 9 columns), ragged ones, one row
@pytest.mark.parametrize("nx,ny,P", [(16, 16, 1), (33, 5, 3), (9, 7, 7), (70, 1, 2), (72, 90, 9), (16, 16, 64), (16, 24, 250), (40, 33, 96)])
@pytest.mark.parametrize("m", [24, 25, 32, 33, 36, 40, 41, 48])
def test_values(lib, nx, ny, P, m):
    print("gram %d x %d, %d problems of %d" % (nx, ny, P, m), flush=True)
    rng = np.random.default_rng(nx * ny + m)
    u = rng.standard_normal((m, 2, ny, nx)) + 1j * rng.standard_normal((m, 2, ny, nx))
    eta = rng.uniform(0.1, 1.0, (ny, nx))
    ref, np_, n = reference(u, eta), m * (m + 1) // 2, 2 * nx * ny
    # all problems on the block of problem 0 (the column list too); the lists: full, one
    # column, and as many as end in each tile
    du, deta, dmap = Dev(lib, u), Dev(lib, eta), Dev(lib, np.zeros(P, np.int32))
    work = Dev(lib, None, nbytes=lib.mxh_gram_work_bytes(m, P))
    lv, bl = Level(nx, ny, 0.1, 0.08), Bloch(np.cos(0.7), np.sin(0.7), np.cos(-1.3), np.sin(-1.3), None, 1, None)
    for mq in [None, m, 1] + list(range(7, m, 8)):
        out = Dev(lib, np.full((P, np_, 4), 7.0))
        a = [C.byref(lv), C.byref(bl), P, dmap.p]
        b = [m, vecs(du, n), deta.p, out.p, work.p]
        cols = np.arange(m)
        if mq is None:
            assert lib.mxh_gram(*a, *b) == 0
        else:
            cols = np.sort(rng.choice(m, mq, replace=False))
            cmap = np.zeros(m + 1, np.int32)
            cmap[0] = mq
            cmap[1:mq + 1] = cols
            dc = Dev(lib, cmap)
            assert lib.mxh_gram_cols(*a, dc.p, *b) == 0
        got = out.get()
        i, j = np.tril_indices(len(cols))
        # sums of nx ny products: below 1e-12 of the Cauchy-Schwarz bound (as the
        # square grids' test); the listed pairs are the first of the output
        for q, r in ((0, ref[0]), (2, ref[1])):
            d = np.sqrt(np.diag(r).real)[cols]
            g = got[:, :len(i), q] + 1j * got[:, :len(i), q + 1]
            err = np.abs(g - r[cols[i], cols[j]]) / (d[i] * d[j])
            assert err.max() <= 1e-12


def test_a_small_grids_wide_block_takes_one_workgroups_time(lib):
    """36 vectors against 24 of one 16^2 problem: the chip is idle, so a launch takes
    its longest workgroup: 6 tile pairs of 3 tiles against 5 pairs of 5.  All 15 pairs
    in each workgroup took 2.5 times as long."""
    best = {}
    rng = np.random.default_rng(1)
    for m in (24, 36):
        u, eta = Dev(lib, rng.standard_normal((m, 512)) + 0j), Dev(lib, np.ones((16, 16)))
        out, work = Dev(lib, None, nbytes=16 * m * (m + 1)), Dev(lib, None, nbytes=lib.mxh_gram_work_bytes(m, 1))
        lv, bl = Level(16, 16, 0.1, 0.1), Bloch(1.0, 0.0, 1.0, 0.0, None, 1, None)
        t = 1.0
        for _ in range(6):
            assert lib.mxh_sync() == 0
            t0 = time.perf_counter()
            for _ in range(200):
                assert lib.mxh_gram(C.byref(lv), C.byref(bl), 1, None, m, vecs(u, 512), eta.p, out.p, work.p) == 0
            assert lib.mxh_sync() == 0
            t = min(t, (time.perf_counter() - t0) / 200)
        best[m] = t
    print("24: %.1f us, 36: %.1f us" % (1e6 * best[24], 1e6 * best[36]))
    assert best[36] <= 1.7 * best[24]
