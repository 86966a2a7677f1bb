"""mxh_curl2: the weighted sum of |curl e_v|^2 / (hx hy) per cell, added to what
the gradient holds, against the sum written out with the Bloch factors.

Tolerance: a cell's term is a sum of four entries, squared (8 roundings), and
nv + 1 terms are added: 20 eps of the largest cell's sum of moduli."""
import ctypes as C

import numpy as np
import pytest

from gpu_abi import Bloch, Dev, Level, Vecs, bind, vecs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    L = bind(M.lib)
    L.mxh_curl2.argtypes = [C.POINTER(Level), C.POINTER(Bloch), C.c_int, Vecs, C.c_void_p, C.c_void_p]
    return L


@pytest.mark.parametrize("nx,ny,nv", [(1, 1, 1), (16, 16, 1), (30, 17, 3), (300, 5, 8)])
def test_curl2_adds_to_the_gradient(lib, nx, ny, nv):
    print("curl2 %d x %d, %d vectors" % (nx, ny, nv), flush=True)
    rng = np.random.default_rng(nx + nv)
    hx, hy, kx, ky = 0.1, 0.07, 1.3, -2.1
    e = rng.standard_normal((nv, 2, ny, nx)) + 1j * rng.standard_normal((nv, 2, ny, nx))
    w, before = rng.uniform(-1.0, 1.0, nv), rng.standard_normal((ny, nx))
    x, y = e[:, 0], e[:, 1]
    xu, yr = np.roll(x, -1, 1), np.roll(y, -1, 2)
    xu[:, -1] *= np.exp(1j * ky)
    yr[:, :, -1] *= np.exp(1j * kx)
    c = np.abs(x - xu - y + yr) ** 2 / (hx * hy)
    scale = np.abs(before) + (np.abs(w)[:, None, None] * 4 * (np.abs(x) + np.abs(xu) + np.abs(y) + np.abs(yr)) ** 2 / (hx * hy)).sum(0)
    lv, bl = Level(nx, ny, hx, hy), Bloch(np.cos(kx), np.sin(kx), np.cos(ky), np.sin(ky), None, 1, None)
    de, dw, dg = Dev(lib, e.reshape(nv, -1)), Dev(lib, w), Dev(lib, before)
    for times in (1, 2):
        assert lib.mxh_curl2(C.byref(lv), C.byref(bl), nv, vecs(de, 2 * nx * ny), dw.p, dg.p) == 0
        ref = before + times * (w[:, None, None] * c).sum(0)
        assert np.abs(dg.get() - ref).max() <= 20 * 2.2e-16 * times * scale.max()
