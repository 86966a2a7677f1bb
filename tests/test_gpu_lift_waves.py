"""The lifting removes the gradient of each of the nine lowest Bloch waves: for
e = G phi_pq (no x) nothing is left of it.  The waves are put in one at a time, so
that a lowest wave that is missing or formed in FP32, or a wrong factor of one
mode, shows in full and not beside the many modes of a random field.

Bounds, relative to e, with every rounding error taken at its worst: waves this
long vary so slowly that errors of neighbouring entries do not average.
g_pq = |(2 pi p + kx) / nx, (2 pi q + ky) / ny| is a wave's gradient, mu_pq about
its square.
- d = G^H M e is formed in FP64 from differences of numbers of the size of e, 3 eps
  |e| an entry; into the lowest wave that is 3 eps / g_00, twice for both parts.
- d is stored and transformed in the multigrid precision: 5 eps a stage, log2 N
  stages; into the lowest of the transform's waves (all but (0, 0)) g_pq / g of it.
- A wave's own factor: 20 eps; the lowest wave's is formed in FP64."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_abi import NONE, Bloch, Dev, Level, Vecs, bind, vecs

pytestmark = pytest.mark.gpu

EPS64, EPS32 = 2.2e-16, 1.2e-7


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny,kx,ky", [(16, 40, 0.3, -1.1), (48, 64, 3.0, 0.2), (128, 128, 0.05, 0.02),
                                         (160, 192, -2.0, 3.0), (512, 256, 0.17, 0.0), (1024, 32, 1.0, -0.4),
                                         (64, 64, 0.0, 0.0)])
def test_gradients_of_the_lowest_waves(prec, nx, ny, kx, ky):
    import maxwell_amd as M
    lib = bind(M.lib)
    lib.mxh_lift_table_bytes.restype = C.c_size_t
    lib.mxh_lift_table.argtypes = [C.c_int, C.POINTER(Level), C.c_void_p]
    lib.mxh_lift.argtypes = [C.c_int, C.POINTER(Level), C.POINTER(Bloch), C.c_int] + [Vecs] * 6 + [C.c_double] + [C.c_void_p] * 3
    print("lift waves prec %d %d x %d k (%g, %g)" % (prec, nx, ny, kx, ky), flush=True)
    dt, eps = (np.complex128, EPS64) if prec == 0 else (np.complex64, EPS32)
    N, h = nx * ny, 1.0 / max(nx, ny)
    g = O.Grid2D(np.ones((ny, nx)), hx=h, hy=1.5 * h, kx=kx, ky=ky)
    i, j = np.arange(nx), np.arange(ny)[:, None]
    waves = [(p, q) for p in (-1, 0, 1) for q in (-1, 0, 1) if (kx, ky) != (0, 0) or (p, q) != (0, 0)]
    e = np.array([O.gradient(g, np.exp(1j * ((2 * np.pi * p + kx) * i / nx + (2 * np.pi * q + ky) * j / ny)).ravel())
                  for p, q in waves])
    nv = len(waves)
    lv = Level(nx, ny, h, 1.5 * h)
    de, dbg, dxg = Dev(lib, e), Dev(lib, np.zeros((nv, N), dt)), Dev(lib, np.zeros((nv, N), dt))
    dcoef, dwork = Dev(lib, np.zeros(2 * nv)), Dev(lib, None, nbytes=8 * 2 * 513 * nv)
    dtab = Dev(lib, None, nbytes=lib.mxh_lift_table_bytes(prec, C.byref(lv)))
    assert lib.mxh_lift_table(prec, C.byref(lv), dtab.p) == 0
    bl = Bloch(np.cos(kx) if kx else 1.0, np.sin(kx), np.cos(ky) if ky else 1.0, np.sin(ky), None, 1, None)
    ev = vecs(de, 2 * N)
    assert lib.mxh_lift(prec, C.byref(lv), C.byref(bl), nv, ev, NONE, vecs(dbg, N), vecs(dxg, N), ev, ev, -1.0, dtab.p,
                        dcoef.p, dwork.p) == 0
    left = np.linalg.norm(de.get(), axis=1) / np.linalg.norm(e, axis=1)
    length = {w: np.hypot((2 * np.pi * w[0] + kx) / nx, (2 * np.pi * w[1] + ky) / ny) for w in waves}
    second = min(v for w, v in length.items() if w != (0, 0))
    for w, r in zip(waves, left):
        bound = 20 * (EPS64 if w == (0, 0) else eps) + 5 * np.log2(N) * eps * length[w] / second
        if (0, 0) in length:
            bound += 6 * EPS64 / length[(0, 0)]
        print("    (%2d, %2d): left %.1e bound %.1e" % (*w, r, bound))
        assert r <= bound
