"""Kernels that hold a whole periodic grid in LDS, against the oracle's
operators in FP64: the smoothing passes of mxh_afw_tile on grids of at most
64 x 64 (rectangular ones and the smallest included) and the coarse end of a
V-cycle in one launch (mxh_edge_cycle, mxh_node_cycle) over one to five
levels, against the same cycle composed from the oracle's sweeps, transfers and
dense solves.

Tolerance: an AFW patch matrix has condition ~8.9 / h^2 (its gradient
direction sees only the mass), so two exact local solves written differently
agree to ~eps / h^2 of the result; the nodal cycle has no such direction
(eps times a few hundred operations)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from gpu_abi import NONE, Bloch, Dev, Level, Vecs, bind, vecs

pytestmark = pytest.mark.gpu

MAXL = 6


class Cycle(C.Structure):
    _fields_ = [("n", C.c_int), ("lv", Level * MAXL), ("eta", C.c_void_p * MAXL), ("b", C.c_void_p * MAXL),
                ("x", C.c_void_p * MAXL)]


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    L = bind(M.lib)
    L.mxh_afw_tile.argtypes = [C.c_int, C.POINTER(Level), C.POINTER(Bloch), C.c_int, Vecs, Vecs, Vecs, C.c_void_p,
                               C.c_int, C.c_int, Vecs, Vecs, Vecs]
    for f in (L.mxh_edge_cycle, L.mxh_node_cycle):
        f.argtypes = [C.c_int, C.POINTER(Cycle), C.POINTER(Bloch), C.c_int, C.c_int, Vecs, Vecs, C.c_int, C.c_void_p,
                      C.c_int]
    L.mxh_coarse_inverse.argtypes = [C.c_int, C.c_int, C.c_void_p, C.c_void_p]
    return L


def rnd(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def random_eta(ny, nx, seed):
    return 1.0 / np.random.default_rng(seed).uniform(1.0, 9.0, size=(ny, nx))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("nx,ny", [(4, 4), (6, 64), (64, 64), (48, 20), (32, 32), (62, 66)])
@pytest.mark.parametrize("mode,nsweep", [(0, 1), (1, 2), (2, 2), (5, 2), (8, 2), (10, 1)])
def test_small_grid_passes(lib, prec, nx, ny, mode, nsweep):
    print("grid pass prec %d %d x %d mode %d x %d" % (prec, nx, ny, mode, nsweep), flush=True)
    rng = np.random.default_rng(nx + 7 * ny + mode)
    h, kx, ky, nv = 1 / 16, 0.7, -1.9, 3
    eta = random_eta(ny, nx, 3)
    g = O.Grid2D(eta, hx=h, hy=0.75 * h, kx=kx, ky=ky)
    E, Ec = 2 * nx * ny, nx * ny // 2
    dt, rt = (np.complex128, np.float64) if prec == 0 else (np.complex64, np.float32)
    b, x, xc = (rnd(rng, nv, k).astype(dt) for k in (E, E, Ec))
    db, dx, dxo, dxc = Dev(lib, b), Dev(lib, x), Dev(lib, np.zeros((nv, E), dt)), Dev(lib, xc)
    dbc, deta = Dev(lib, np.zeros((nv, Ec), dt)), Dev(lib, eta.astype(rt))
    lv, bl = Level(nx, ny, h, 0.75 * h), Bloch(np.cos(kx), np.sin(kx), np.cos(ky), np.sin(ky), None, 1, None)
    res = mode & 8
    assert lib.mxh_afw_tile(prec, C.byref(lv), C.byref(bl), nv, vecs(db, E), vecs(dx, E), vecs(dxo, E), deta.p, nsweep,
                            mode, vecs(dxc, Ec) if mode & 4 else NONE, vecs(dbc, Ec) if res else NONE,
                            vecs(dxc, Ec) if res else NONE) == 0
    tol = (2e-15 if prec == 0 else 1e-6) / (h * h)
    got = dxo.get()
    for v in range(nv):
        ref = np.zeros(E, complex) if mode & 2 else x[v].astype(complex)
        if mode & 4:
            ref = O.prolong_edge(g, xc[v].astype(complex), ref)
        for _ in range(nsweep):
            ref = O.gs_edge(g, b[v].astype(complex), ref, backward=bool(mode & 1), colour_order=1)
        assert np.abs(got[v] - ref).max() <= tol * np.abs(ref).max(), v
        if res:
            xs = ref if prec == 0 else got[v].astype(complex)
            rc = O.restrict_edge(g, O.addeval(g, -1.0, -1.0, xs, b[v].astype(complex)))
            scale = np.abs(rc).max() if prec == 0 else np.abs(O.restrict_edge(g, O.addeval(g, 1.0, 1.0, xs))).max()
            assert np.abs(dbc.get()[v] - rc).max() <= tol * scale
            assert np.abs(dxc.get()[v]).max() == 0


def hierarchy(nx0, ny0, levels, h, kx, ky, seed):
    """Grids of levels 0 .. levels - 1, the finest with a random eta."""
    nx, ny = nx0 << (levels - 1), ny0 << (levels - 1)
    gs = [O.Grid2D(random_eta(ny, nx, seed), hx=h, hy=1.25 * h, kx=kx, ky=ky)]
    for _ in range(levels - 1):
        e = gs[0].eta
        e = 0.25 * (e[::2, ::2] + e[::2, 1::2] + e[1::2, ::2] + e[1::2, 1::2])
        gs.insert(0, O.Grid2D(e, hx=2 * gs[0].hx, hy=2 * gs[0].hy, kx=kx, ky=ky))
    return gs


def oracle_cycle(gs, node, l, b, x, nu, A0, lower):
    g = gs[l]
    if l == 0:
        x = np.linalg.solve(A0, b)
        lower[0] = (b, x)
        return x
    sweep = O.gs_node if node else O.gs_edge
    for _ in range(nu):
        x = sweep(g, b, x, backward=False, colour_order=1)
    r = b - O.addeval_node(g, 1.0, x) if node else O.addeval(g, -1.0, -1.0, x, b)
    bc = O.restrict_node(g, r) if node else O.restrict_edge(g, r)
    xc = oracle_cycle(gs, node, l - 1, bc, np.zeros_like(bc), nu, A0, lower)
    x = O.prolong_node(g, xc, x) if node else O.prolong_edge(g, xc, x)
    for _ in range(nu):
        x = sweep(g, b, x, backward=True, colour_order=1)
    lower[l] = (b, x)
    return x


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("node", [False, True])
@pytest.mark.parametrize("nx0,ny0,levels,nu,xzero", [(4, 4, 4, 2, 1), (4, 4, 1, 2, 1), (2, 2, 5, 1, 0), (6, 4, 3, 2, 0),
                                                     (8, 8, 3, 3, 1), (4, 8, 2, 2, 0)])
def test_coarse_cycle(lib, prec, node, nx0, ny0, levels, nu, xzero):
    print("cycle prec %d node %d %d x %d, %d levels" % (prec, node, nx0, ny0, levels), flush=True)
    rng = np.random.default_rng(nx0 + ny0 + levels)
    h, ks, nv = 1 / 32, [(0.4, -2.2), (np.pi, 1.1)], 3
    hs = [hierarchy(nx0, ny0, levels, h, kx, ky, 5) for kx, ky in ks]
    gs, comp = hs[0], 1 if node else 2
    dt, rt = (np.complex128, np.float64) if prec == 0 else (np.complex64, np.float32)
    n, n0 = comp * gs[-1].nx * gs[-1].ny, comp * nx0 * ny0
    # the inverse of each problem's coarsest matrix from its Cholesky factor (column-major)
    A0 = [O.dense_node(q[0], fixnull=True) if node else O.dense_edge(q[0], 1.0, 1.0) for q in hs]
    L = np.stack([np.linalg.cholesky(a).T for a in A0])
    dL, dW = Dev(lib, L), Dev(lib, np.zeros((2, n0, n0), complex))
    assert lib.mxh_coarse_inverse(n0, 2, dL.p, dW.p) == 0
    W = dW.get()
    for p in range(2):
        assert np.abs(W[p] @ A0[p] - np.eye(n0)).max() < 1e-15 * n0 * np.linalg.cond(A0[p])
    cy = Cycle(levels)
    detas = [Dev(lib, q.eta.astype(rt)) for q in gs]
    for l, q in enumerate(gs):
        cy.lv[l] = Level(q.nx, q.ny, q.hx, q.hy)
        cy.eta[l] = None if node else detas[l].p
    assert lib.mxh_cycle_supported(prec, C.byref(cy)) == 1
    # vectors 0, 1 of problem 1, vector 2 of problem 0 (vpp 2), b of the edge cycle through a map
    gmap = np.array([2, 3, 0], np.int32)
    bmap = np.array([1, 3, 0], np.int32)
    bf = np.array([[np.cos(a), np.sin(a), np.cos(c), np.sin(c)] for a, c in ks])
    dg, dm, dbf = Dev(lib, gmap), Dev(lib, bmap), Dev(lib, bf)
    b, x = rnd(rng, 4, n).astype(dt), rnd(rng, nv, n).astype(dt)
    db, dx = Dev(lib, b), Dev(lib, x)
    bl = Bloch(1, 0, 1, 0, dbf.p, 2, dg.p)
    run = lib.mxh_node_cycle if node else lib.mxh_edge_cycle
    bv = vecs(db, n)
    if not node:
        bv.map = dm.p
    assert run(prec, C.byref(cy), C.byref(bl), nv, nu, bv, vecs(dx, n), xzero, dW.p, 1) == 0
    got = dx.get()
    eps = 2.2e-16 if prec == 0 else 1.2e-7
    tol = 500 * eps if node else 10 * eps / (h * h)
    for v in range(nv):
        p = int(gmap[v]) // 2
        bb = b[v if node else bmap[v]].astype(complex)
        ref = oracle_cycle(hs[p], node, levels - 1, bb, np.zeros(n, complex) if xzero else x[v].astype(complex), nu,
                           A0[p], {})
        err = np.abs(got[v] - ref).max() / np.abs(ref).max()
        print("    vector %d rel err %.2e (tol %.2e)" % (v, err, tol))
        assert err <= tol
    # one vector with the lower levels returned
    if levels > 1:
        dlow = [(Dev(lib, np.zeros(comp * q.nx * q.ny, dt)), Dev(lib, np.zeros(comp * q.nx * q.ny, dt))) for q in gs[:-1]]
        for l, (p, q) in enumerate(dlow):
            cy.b[l], cy.x[l] = p.p, q.p
        dx1 = Dev(lib, x[:1])
        b1 = Bloch(np.cos(ks[0][0]), np.sin(ks[0][0]), np.cos(ks[0][1]), np.sin(ks[0][1]), None, 1, None)
        assert run(prec, C.byref(cy), C.byref(b1), 1, nu, vecs(db, n), vecs(dx1, n), xzero, dW.p, 0) == 0
        low = {}
        oracle_cycle(hs[0], node, levels - 1, b[0].astype(complex),
                     np.zeros(n, complex) if xzero else x[0].astype(complex), nu, A0[0], low)
        for l, (p, q) in enumerate(dlow):
            for d, ref in ((p, low[l][0]), (q, low[l][1])):
                assert np.abs(d.get() - ref).max() <= 50 * tol * max(np.abs(low[l][0]).max(), np.abs(low[l][1]).max())
        # lower levels only for a single vector
        assert run(prec, C.byref(cy), C.byref(b1), 2, nu, vecs(db, n), vecs(dx1, n), xzero, dW.p, 0) != 0
