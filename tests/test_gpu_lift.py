"""The direct gradient lifting (mxh_lift): out = u - x + alpha G xg with the node
system A xg = G^H M (e - x) solved by transforms.  With u = e and alpha = -1
the result is fixed by two properties, checked with the oracle's operators:
out differs from w = e - x by a gradient (the same curl in every cell), and it
is divergence-free (G^H M out = 0).  Grids of one launch (the vector in LDS),
of row and column passes, with an odd radix and with nx != ny; the Gamma
point; a point next to it, where the lowest wave's eigenvalue is ~1e-7.

Tolerances.  The solve leaves an error of a few eps in the gradient it
subtracts (relative to it in the energy norm, log2 n stages), amplified on
the lowest modes but one (mu ~ (2 pi / n)^2 / 4 of the largest, in whose
square root the gradient error grows) to about eps n: G^H M out is
compared with |M| |w| at 50 eps n."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_abi import NONE, Bloch, Dev, Level, Vecs, bind, vecs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    L = bind(M.lib)
    L.mxh_lift_table_bytes.restype = C.c_size_t
    L.mxh_lift_table.argtypes = [C.c_int, C.POINTER(Level), C.c_void_p]
    L.mxh_lift.argtypes = [C.c_int, C.POINTER(Level), C.POINTER(Bloch), C.c_int, Vecs, Vecs, Vecs, Vecs, Vecs, Vecs,
                           C.c_double, C.c_void_p, C.c_void_p, C.c_void_p]
    return L


CASES = [(8, 8, 0.3, -1.1), (16, 40, 0.0, 0.0), (48, 64, np.pi, 0.2), (128, 128, 0.05, 0.0), (160, 192, -2.0, 3.0),
         (256, 320, 0.0, 0.0), (512, 256, 0.17, 0.0), (1024, 32, 1.0, -0.4)]


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny,kx,ky", CASES)
@pytest.mark.parametrize("form", ["in place", "correction only", "no x"])
def test_lift_is_divergence_free(lib, prec, nx, ny, kx, ky, form):
    print("lift prec %d %d x %d k (%g, %g) %s" % (prec, nx, ny, kx, ky, form), flush=True)
    h = 1.0 / max(nx, ny)
    g = O.Grid2D(np.ones((ny, nx)), hx=h, hy=1.5 * h, kx=kx, ky=ky)
    lv = Level(nx, ny, h, 1.5 * h)
    assert lib.mxh_lift_supported(prec, C.byref(lv)) == 1
    N, nv = nx * ny, 2
    rng = np.random.default_rng(nx + 3 * ny)
    dt = np.complex128 if prec == 0 else np.complex64
    e = rng.standard_normal((nv, 2 * N)) + 1j * rng.standard_normal((nv, 2 * N))
    x = (0.3 * (rng.standard_normal((nv, 2 * N)) + 1j * rng.standard_normal((nv, 2 * N)))).astype(dt)
    de, dx = Dev(lib, e), None if form == "no x" else Dev(lib, x)
    dbg, dxg = Dev(lib, np.zeros((nv, N), dt)), Dev(lib, np.zeros((nv, N), dt))
    dout = Dev(lib, np.zeros((nv, 2 * N), complex))
    dcoef, dwork = Dev(lib, np.zeros(2 * nv)), Dev(lib, None, nbytes=8 * 2 * 513 * nv)
    dtab = Dev(lib, None, nbytes=lib.mxh_lift_table_bytes(prec, C.byref(lv)))
    assert lib.mxh_lift_table(prec, C.byref(lv), dtab.p) == 0
    bl = Bloch(np.cos(kx) if kx else 1.0, np.sin(kx), np.cos(ky) if ky else 1.0, np.sin(ky), None, 1, None)
    inplace = form != "correction only"
    ev = vecs(de, 2 * N)
    assert lib.mxh_lift(prec, C.byref(lv), C.byref(bl), nv, ev, vecs(dx, 2 * N), vecs(dbg, N), vecs(dxg, N),
                        ev if inplace else NONE, ev if inplace else vecs(dout, 2 * N), -1.0, dtab.p, dcoef.p,
                        dwork.p) == 0
    got = de.get() if inplace else dout.get() + e
    eps = 2.2e-16 if prec == 0 else 1.2e-7
    for v in range(nv):
        w = e[v] if form == "no x" else e[v] - x[v].astype(complex)
        mw = O.addeval(g, 0.0, 1.0, w)
        div = O.adjgradient(g, O.addeval(g, 0.0, 1.0, got[v]))
        curl = O.addeval(g, 1.0, 0.0, got[v] - w)
        d, c = np.abs(div).max() / np.abs(mw).max(), np.abs(curl).max() / np.abs(O.addeval(g, 1.0, 0.0, w)).max()
        print("    divergence %.2e curl change %.2e" % (d, c))
        assert d <= 50 * eps * max(nx, ny)
        assert c <= 50 * eps * max(nx, ny)


def test_lift_refuses_unsupported_grids(lib):
    lv = Level(14, 14, 1 / 14, 1 / 14)
    assert lib.mxh_lift_supported(0, C.byref(lv)) == 0
    bl = Bloch(1.0, 0.0, 1.0, 0.0, None, 1, None)
    assert lib.mxh_lift(0, C.byref(lv), C.byref(bl), 1, NONE, NONE, NONE, NONE, NONE, NONE, -1.0, None, None,
                        None) != 0
