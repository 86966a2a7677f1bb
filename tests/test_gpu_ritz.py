"""The device Rayleigh-Ritz eigenproblems (mxh_ritz) against scipy's generalised
eigensolver: block sizes from 1 to the largest (48 columns), odd and even,
column lists with gaps, degenerate eigenvalues, columns that depend on earlier
ones, and the statuses for sums that are not finite or not definite.

The pencils are built from random unit columns, B = X^H X with condition of a
few hundred at most, so eigenvalues agree to eps times that and the size."""
import ctypes as C

import numpy as np
import pytest
import scipy.linalg as sl

from gpu_abi import Dev, bind

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import maxwell_amd as M
    L = bind(M.lib)
    L.mxh_ritz.argtypes = [C.c_int, C.c_int, C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_double, C.c_double,
                           C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    return L


def pencil(n, rng, degenerate=False):
    """(K, M) of n random columns over 3 n + 40 unknowns, K with eigenvalues from 0.5 to 2000."""
    N = 3 * n + 40
    X = rng.standard_normal((N, n)) + 1j * rng.standard_normal((N, n))
    X *= 10.0 ** rng.uniform(-3, 3, n)  # columns of any size
    d = np.geomspace(0.5, 2000.0, N)
    if degenerate:
        d[:] = np.repeat(np.geomspace(0.5, 2000.0, (N + 4) // 5), 5)[:N]
    return X.conj().T @ (d[:, None] * X), X.conj().T @ X


def pack(K, Mm, k, sk):
    """Gram sums of pairs a >= b in the layout of mxh_gram for k columns."""
    n = K.shape[0]
    out = np.full((k * (k + 1) // 2, 4), np.nan)
    for a in range(n):
        for b in range(a + 1):
            out[a * (a + 1) // 2 + b] = [K[a, b].real / sk, K[a, b].imag / sk, Mm[a, b].real, Mm[a, b].imag]
    return out


def run(lib, m, basis, grams, lists, sk, pivot):
    P, k = len(grams), basis or m
    pmap = np.arange(P)[::-1].astype(np.int32).copy()
    dg, dp = Dev(lib, np.stack(grams)), Dev(lib, pmap)
    cm = np.zeros((P, k + 1), np.int32)
    for j, lst in enumerate(lists):
        cm[pmap[j], 0], cm[pmap[j], 1:1 + len(lst)] = len(lst), lst
    dcm = Dev(lib, cm)
    dC = Dev(lib, np.full((P, 2 * m if basis else m, k), 7.0 + 0j))
    dl, ds = Dev(lib, np.zeros((P, k))), Dev(lib, np.full(P, 9, np.int32))
    assert lib.mxh_ritz(m, basis, P, dp.p, dcm.p if basis else None, dg.p, sk, pivot, dC.p, dl.p, k, ds.p) == 0
    return dC.get().transpose(0, 2, 1), dl.get()[pmap], ds.get()


def check(K, Mm, cols, m, c, lam):
    """c: coefficients (k x m) of a problem whose listed columns have the pencil (K, Mm)."""
    ref = sl.eigh(K + Mm, Mm, eigvals_only=True)[:m]
    assert np.abs(lam - ref).max() <= 1e-11 * np.abs(ref).max() and (np.diff(lam) >= 0).all()
    rest = np.setdiff1d(np.arange(c.shape[0]), cols)
    assert not c[rest].any()
    x = c[cols]
    assert np.abs(x.conj().T @ Mm @ x - np.eye(m)).max() <= 1e-11
    assert np.abs(x.conj().T @ (K + Mm) @ x - np.diag(lam)).max() <= 1e-11 * np.abs(lam).max()


@pytest.mark.parametrize("m", [1, 2, 5, 10, 12, 17, 32])
@pytest.mark.parametrize("degenerate", [False, True])
def test_block_problems(lib, m, degenerate):
    print("ritz block %d" % m, flush=True)
    rng = np.random.default_rng(m)
    ps = [pencil(m, rng, degenerate) for _ in range(3)]
    Cm, lam, st = run(lib, m, 0, [pack(K, Mm, m, 16.0) for K, Mm in ps], [[]] * 3, 16.0, 1e-13)
    assert (st == 0).all()
    for j, (K, Mm) in enumerate(ps):
        check(K, Mm, np.arange(m), m, Cm[j], lam[j][:m])


@pytest.mark.parametrize("m", [1, 2, 7, 12, 16])
def test_listed_columns(lib, m):
    print("ritz basis of %d" % (3 * m), flush=True)
    rng = np.random.default_rng(30 + m)
    k = 3 * m
    lists = [np.arange(k), np.arange(m), np.r_[np.arange(m), m + np.flatnonzero(rng.random(2 * m) < 0.6)]]
    ps = [pencil(len(c), rng) for c in lists]
    Cm, lam, st = run(lib, m, k, [pack(K, Mm, k, 4.0) for K, Mm in ps], lists, 4.0, 1e-7)
    assert (st == 0).all()
    for j, ((K, Mm), cols) in enumerate(zip(ps, lists)):
        e, p = Cm[j][:, :m], Cm[j][:, m:]
        check(K, Mm, cols, m, e, lam[j][:m])
        assert not p[:m].any() and np.array_equal(p[m:], e[m:])


def test_dependent_columns_and_statuses(lib):
    rng = np.random.default_rng(5)
    m, k = 4, 12
    N = 60
    X = rng.standard_normal((N, k)) + 1j * rng.standard_normal((N, k))
    X[:, 6] = X[:, :3] @ [1.0, 2j, -1.0]  # dependent on the block
    X[:, 9] = 0.0
    d = np.geomspace(0.5, 300.0, N)
    K, Mm = X.conj().T @ (d[:, None] * X), X.conj().T @ X
    good = pack(K, Mm, k, 1.0)
    few = X.copy()
    few[:, 3:] = few[:, :1] * np.arange(1, 10)  # rank 3 < m
    bad = good.copy()
    bad[7, 2] = np.inf
    Cm, lam, st = run(lib, m, k, [good, pack(few.conj().T @ (d[:, None] * few), few.conj().T @ few, k, 1.0), bad, good],
                      [np.arange(k)] * 4, 1.0, 1e-7)
    assert st.tolist() == [0, 2, 1, 0]
    assert not Cm[1].any() and not Cm[2].any()
    keep = np.setdiff1d(np.arange(k), [6, 9])
    for j in (0, 3):
        check(K[np.ix_(keep, keep)], Mm[np.ix_(keep, keep)], keep, m, Cm[j][:, :m], lam[j][:m])
    # a block with a repeated vector is not definite
    Xb = X[:, :5].copy()
    Xb[:, 4] = Xb[:, 1]
    _, _, st = run(lib, 5, 0, [pack(Xb.conj().T @ (d[:, None] * Xb), Xb.conj().T @ Xb, 5, 1.0)], [[]], 1.0, 1e-13)
    assert st[0] == 2
