"""Row bands of the Gram sums where the partial sums' buffer (2048 sets, fewer in
the static scratch of wide blocks) sets their height: tall grids and many
problems.  A launch has to keep the chip as busy as on a grid of the same cells
that needs no tall bands; values against the sums written out."""
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


def setup(lib, nx, ny, P, m, seed=0):
    """All P problems on one block of vectors: the map sends them to problem 0."""
    rng = np.random.default_rng(seed)
    u = rng.standard_normal((m, 2 * nx * ny)) + 1j * rng.standard_normal((m, 2 * nx * ny))
    eta = rng.uniform(0.1, 1.0, (ny, nx))
    np_ = m * (m + 1) // 2
    return dict(u=u, eta=eta, du=Dev(lib, u), deta=Dev(lib, eta), dmap=Dev(lib, np.zeros(P, np.int32)),
                out=Dev(lib, np.zeros((P, np_, 4))), work=Dev(lib, None, nbytes=lib.mxh_gram_work_bytes(m, P)),
                lv=Level(nx, ny, 0.1, 0.08), bl=Bloch(np.cos(0.7), np.sin(0.7), np.cos(-1.3), np.sin(-1.3), None, 1, None))


def gram(lib, s, P, m, static):
    n = s["u"].shape[1]
    a = [C.byref(s["lv"]), C.byref(s["bl"]), P, s["dmap"].p, m, vecs(s["du"], n), s["deta"].p, s["out"].p]
    assert (lib.mxh_gram_static(*a) if static else lib.mxh_gram(*a, s["work"].p)) == 0


# least heights of 64 and 129 rows, one band a problem (70 rows), the static
# scratch's 222 sets of 48 columns (116 rows), 26 rows with a ragged last band
@pytest.mark.parametrize("nx,ny,P,m,static", [(16, 3907, 33, 3, False), (24, 2049, 128, 2, False), (40, 70, 2048, 1, False),
                                              (9, 1500, 16, 48, True), (32, 1301, 40, 5, False)])
def test_values(lib, nx, ny, P, m, static):
    print("gram %d x %d, %d problems of %d" % (nx, ny, P, m), flush=True)
    s = setup(lib, nx, ny, P, m, nx)
    gram(lib, s, P, m, static)
    got = s["out"].get()
    u = s["u"].reshape(m, 2, ny, nx)
    x, y = u[:, 0], u[:, 1]
    xu, yr = np.roll(x, -1, 1), np.roll(y, -1, 2)
    xu[:, -1] *= np.exp(-1.3j)
    yr[:, :, -1] *= np.exp(0.7j)
    c = (x - xu - y + yr).reshape(m, -1)
    K = c.conj() @ (s["eta"].ravel() * c).T
    mx, my = 0.08 / 0.1 / 6.0, 0.1 / 0.08 / 6.0
    f = lambda a, b: a.reshape(m, -1).conj() @ b.reshape(m, -1).T
    Mm = mx * (4 * f(x, x) + f(x, xu) + f(xu, x)) + my * (4 * f(y, y) + f(y, yr) + f(yr, y))
    a, b = np.tril_indices(m)
    # sums of nx ny products: the rounding of numpy's and of the kernel's partial
    # sums, below 1e-12 of the Cauchy-Schwarz bound (as the square grids' test)
    for q, ref in ((0, K), (2, Mm)):
        d = np.sqrt(np.diag(ref).real)
        err = np.abs(got[:, :, q] + 1j * got[:, :, q + 1] - ref[a, b]) / (d[a] * d[b])
        assert err.max() <= 1e-12


@pytest.mark.parametrize("tall,wide,P,m,static", [((64, 8192), (1024, 512), 20, 8, False),
                                                  ((256, 4096), (1024, 1024), 33, 12, False),
                                                  ((256, 2048), (1024, 512), 16, 36, True)])
def test_tall_grids_are_no_slower(lib, tall, wide, P, m, static):
    best = []
    for nx, ny in (tall, wide):
        s = setup(lib, nx, ny, P, m)
        gram(lib, s, P, m, static)
        t = 1.0
        for _ in range(5):
            assert lib.mxh_sync() == 0
            t0 = time.perf_counter()
            gram(lib, s, P, m, static)
            assert lib.mxh_sync() == 0
            t = min(t, time.perf_counter() - t0)
        best.append(t)
    print("%s %.2f ms, %s %.2f ms" % (tall, 1e3 * best[0], wide, 1e3 * best[1]))
    # the same cells; a band costs one row more than it holds, and the last round
    # of workgroups may be nearly empty on one side
    assert best[0] <= 2.0 * best[1]
