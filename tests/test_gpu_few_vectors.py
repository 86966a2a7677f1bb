"""The tile-fused smoothers on both sides of the rule that gives small launches
small tiles (512 tiles of 12 x 12 owned nodes; one vector always), against the
oracle's sweeps, transfers and residuals in FP64.

Tolerances as the whole grids': an AFW patch matrix has condition ~8.9 / h^2,
so two exact local solves written differently agree to ~eps / h^2 of the
result; the nodal sweeps have no such direction."""
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
    L.mxh_afw_tile.argtypes = [C.c_int, C.POINTER(Level), C.POINTER(Bloch), C.c_int, Vecs, Vecs, Vecs, C.c_void_p,
                               C.c_int, C.c_int, Vecs, Vecs, Vecs]
    L.mxh_node_tile.argtypes = [C.c_int, C.POINTER(Level), C.POINTER(Bloch), C.c_int, Vecs, Vecs, Vecs, C.c_int,
                                C.c_int, Vecs, Vecs, Vecs]
    return L


# 64 x 64: 36 tiles a vector (14: 504, 15: 540); 34 x 36: 3 x 3; 6 x 258: a side
# that wraps several times within a region; 24 x 72: whole tiles; 150 x 162
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny,nv", [(64, 64, 14), (64, 64, 15), (34, 36, 3), (6, 258, 2), (24, 72, 1), (150, 162, 1)])
@pytest.mark.parametrize("node", [False, True])
@pytest.mark.parametrize("mode,nsweep", [(0, 1), (1, 2), (2, 2), (5, 2), (8, 2), (10, 1)])
def test_small_launches(lib, prec, nx, ny, nv, node, mode, nsweep):
    print("prec %d %d x %d, %d vectors, node %d, mode %d x %d" % (prec, nx, ny, nv, node, mode, nsweep), flush=True)
    rng = np.random.default_rng(nx + 7 * ny + mode)
    h, ks = 1 / 16, [(0.7, -1.9), (np.pi, 2.2)]
    eta = 1.0 / rng.uniform(1.0, 9.0, size=(ny, nx))
    gs = [O.Grid2D(eta, hx=h, hy=0.75 * h, kx=kx, ky=ky) for kx, ky in ks]
    E, Ec = (nx * ny, nx * ny // 4) if node else (2 * nx * ny, nx * ny // 2)
    dt, rt = (np.complex128, np.float64) if prec == 0 else (np.complex64, np.float32)
    b, x, xc = ((rng.standard_normal((nv, k)) + 1j * rng.standard_normal((nv, k))).astype(dt) for k in (E, E, Ec))
    db, dx, dxo, dxc = Dev(lib, b), Dev(lib, x), Dev(lib, np.zeros((nv, E), dt)), Dev(lib, xc)
    dbc, deta = Dev(lib, np.zeros((nv, Ec), dt)), Dev(lib, eta.astype(rt))
    # the last vector is of the second problem
    vmap = np.array([0] * (nv - 1) + [1], np.int32)
    dmap, dbf = Dev(lib, vmap), Dev(lib, np.array([[np.cos(a), np.sin(a), np.cos(c), np.sin(c)] for a, c in ks]))
    lv, bl = Level(nx, ny, h, 0.75 * h), Bloch(1, 0, 1, 0, dbf.p, 1, dmap.p)
    res = mode & 8
    args = [nsweep, mode, vecs(dxc, Ec) if mode & 4 else NONE, vecs(dbc, Ec) if res else NONE,
            vecs(dxc, Ec) if res else NONE]
    head = [prec, C.byref(lv), C.byref(bl), nv, vecs(db, E), vecs(dx, E), vecs(dxo, E)]
    assert (lib.mxh_node_tile(*head, *args) if node else lib.mxh_afw_tile(*head, deta.p, *args)) == 0
    if node:
        tol = 200 * (2.2e-16 if prec == 0 else 1.2e-7)
    else:
        tol = (2e-15 if prec == 0 else 1e-6) / (h * h)
    sweep = O.gs_node if node else O.gs_edge
    got, gotb, gotx = dxo.get(), dbc.get(), dxc.get()
    for v in sorted({0, nv // 2, nv - 1}):
        g = gs[vmap[v]]
        bb = b[v].astype(complex)
        ref = np.zeros(E, complex) if mode & 2 else x[v].astype(complex)
        if mode & 4:
            ref = (O.prolong_node if node else O.prolong_edge)(g, xc[v].astype(complex), ref)
        for _ in range(nsweep):
            ref = sweep(g, bb, ref, backward=bool(mode & 1), colour_order=1)
        assert np.abs(got[v] - ref).max() <= tol * np.abs(ref).max(), v
        if res:
            xs = ref if prec == 0 else got[v].astype(complex)
            if node:
                op = lambda y: O.restrict_node(g, y)
                r, a = bb - O.addeval_node(g, 1.0, xs), O.addeval_node(g, 1.0, xs)
            else:
                op = lambda y: O.restrict_edge(g, y)
                r, a = O.addeval(g, -1.0, -1.0, xs, bb), O.addeval(g, 1.0, 1.0, xs)
            rc = op(r)
            scale = np.abs(rc).max() if prec == 0 else np.abs(op(a)).max()
            assert np.abs(gotb[v] - rc).max() <= tol * scale, v
            assert np.abs(gotx[v]).max() == 0
