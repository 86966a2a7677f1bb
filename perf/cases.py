"""What a program built on this library has it do, as measurable cases.

Four cases go through the batched solver (whole band-structure solves and the
adjoint that follows one), five through the device C-ABI that a block step is
made of, three through the reference's module API that its drivers link
against.  listed() holds the workloads of the benchmark and of the tests at
their own sizes; draw() gives further cases of the same ranges (grids of 16 to
512 intervals, square and not, powers of two and not, blocks of 2 to 16
vectors, 1 to 64 Bloch problems, both precisions, both methods).

Device arrays are torch tensors (or views of the library's own vectors), made
from the seed alone.  The library launches on a stream of its own, so every
prepare() ends with a device synchronisation.
"""
import ctypes as C
import math

import numpy as np
import torch

import maxwell_amd as mx

F64, F32 = 0, 1
D, CD = torch.float64, torch.complex128
LIB = mx.lib


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # The headline workload: the band structure of a rod on 512 x 512 cells,
        # 64 k-points on Gamma-X-M-Gamma in one batch, 10 bands, LOBPCG with the
        # FP32 multigrid; the largest solve of a production scan.
        dict(name="path_512_mixed", kind="solve", n0=4, levels=7, pattern="rod", ks="path", problems=64, block=12,
             neig=10, method="lobpcg", prec=F32, autotune=True),
        # One launch group of a Brillouin-zone surface: 64 neighbouring points of
        # the 32 x 32 k-grid on a 256 x 256 supercell, 8 bands, block PINVIT.
        dict(name="surface_256_mixed", kind="solve", n0=4, levels=6, pattern="supercell", ks="zone", problems=64,
             block=10, neig=8, method="pinvit", prec=F32, autotune=True),
        # A quick look at a small cell in plain FP64: 64 x 64, 16 k-points; the
        # launches and the host's Ritz step weigh as much as the kernels.
        dict(name="path_64_f64", kind="solve", n0=4, levels=4, pattern="rod", ks="path", problems=16, block=12,
             neig=10, method="pinvit", prec=F64, autotune=False),
        # Band-gap optimisation: the gradient of one band with respect to every
        # cell's 1/eps after a solve on the 256 x 256 random medium.
        dict(name="gradient_256", kind="gradient", n0=4, levels=6, first=0, count=1, block=8, neig=4),
        # The block step's layers on the 512 x 512 grid, at the half-batch
        # launches of the headline solve or a part of them: the Gram sums of
        # [E W P] with a third of the vectors locked,
        dict(name="gram_512", kind="gram", nx=512, ny=512, m=36, cols=32, problems=16),
        # the defects and their norms (FP64 vectors, FP32 right-hand sides),
        dict(name="defect_512", kind="defect", nx=512, ny=512, nv=192, prec=F32),
        # the gradient lifting's right-hand side and update,
        dict(name="lift_512", kind="lift", nx=512, ny=512, nv=192, prec=F32),
        # and the update of the block and its search directions.
        dict(name="update_512", kind="update", nx=512, ny=512, m=12, problems=16),
        # The edge smoother's passes of a V(2,2) cycle (down with residual and
        # restriction, up with prolongation) in FP64 at the surface's grid.
        dict(name="smooth_256_f64", kind="smooth", nx=256, ny=256, nv=96),
        # The drivers' inner loop: one PINVIT step of one vector through the
        # module API (2 edge V-cycles, 5 nodal ones) at 256 x 256.
        dict(name="vector_step_256", kind="vector_step", n0=4, levels=6, prec_steps=2, gradient_steps=5),
        # The drivers' Ritz matrices, entry by entry, on their smallest grid:
        # the smallest calls of all, an energy and a mass product per pair.
        dict(name="ritz_rows_32", kind="ritz_rows", nx=32, ny=32, vectors=4),
        # The drivers' M-orthonormalisation of an extrapolated basis (two
        # sources of 12 vectors).
        dict(name="orthonormalize_128", kind="orthonormalize", nx=128, ny=128, vectors=24),
    ]


def _size(rng, lo, hi):
    """An even number of intervals, spread over the logarithm of the range."""
    return max(lo, 2 * int(round(0.5 * math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _grid(rng, lo, hi):
    nx = _size(rng, lo, hi)
    return nx, nx if rng.random() < 0.4 else _size(rng, lo, hi)


def _count(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "gradient", "gram", "defect", "lift", "update", "smooth", "vector_step",
                       "ritz_rows", "orthonormalize"])
    if kind == "solve":
        # grids of 16 to 256 (also 3 2^k), the smaller the more of them per batch
        n0 = rng.choice([4, 4, 6])
        levels = rng.randint(2, 6 if n0 == 4 else 5)
        block = rng.choice([6, 8, 9, 10, 12])
        return dict(kind=kind, n0=n0, levels=levels, pattern=rng.choice(["rod", "supercell"]),
                    ks=rng.choice(["path", "zone"]), problems=_count(rng, 1, 32 if levels < 6 else 12), block=block,
                    neig=block - 2, method=rng.choice(["lobpcg", "pinvit"]), prec=rng.choice([F64, F32]),
                    autotune=levels > 4 and rng.random() < 0.5)
    if kind == "gradient":
        return dict(kind=kind, n0=4, levels=rng.randint(3, 6), first=0, count=rng.choice([1, 2]),
                    block=rng.choice([6, 7, 8]), neig=4)
    if kind == "gram":
        nx, ny = _grid(rng, 16, 512)
        m = rng.choice([5, 8, 10, 12, 16, 24, 30, 36, 48])
        cols = m if m < 24 or m % 3 else m - rng.randint(0, m // 3)
        problems = min(_count(rng, 1, 64), max(1, int(16 * 36 * 512 * 512 / (m * nx * ny))))
        return dict(kind=kind, nx=nx, ny=ny, m=m, cols=cols, problems=problems)
    if kind in ("defect", "lift", "smooth"):
        nx, ny = _grid(rng, 16, 512)
        nv = min(_count(rng, 1, 768), max(1, int((96 if kind == "smooth" else 384) * 256 * 256 / (nx * ny))))
        case = dict(kind=kind, nx=nx, ny=ny, nv=nv)
        if kind != "smooth":
            case["prec"] = rng.choice([F64, F32])
        return case
    if kind == "update":
        nx, ny = _grid(rng, 16, 512)
        m = rng.choice([2, 4, 6, 8, 10, 12, 16])
        problems = min(_count(rng, 1, 64), max(1, int(16 * 12 * 512 * 512 / (m * nx * ny))))
        return dict(kind=kind, nx=nx, ny=ny, m=m, problems=problems)
    if kind == "vector_step":
        n0 = rng.choice([4, 6])
        return dict(kind=kind, n0=n0, levels=rng.randint(2, 6 if n0 == 4 else 5), prec_steps=rng.choice([1, 2]),
                    gradient_steps=rng.choice([2, 5]))
    nx, ny = _grid(rng, 16, 256)
    return dict(kind=kind, nx=nx, ny=ny, vectors=rng.randint(2, 6 if kind == "ritz_rows" else 36))


# ------------------------------------------------------------------ the library's C types
class Level(C.Structure):
    _fields_ = [("nx", C.c_int), ("ny", C.c_int), ("hx", C.c_double), ("hy", C.c_double)]


class Bloch(C.Structure):
    _fields_ = [("xr", C.c_double), ("xi", C.c_double), ("yr", C.c_double), ("yi", C.c_double),
                ("per_problem", C.c_void_p), ("vpp", C.c_int), ("vmap", C.c_void_p)]


class Vecs(C.Structure):
    _fields_ = [("p", C.c_void_p), ("stride", C.c_longlong), ("map", C.c_void_p)]


_LV, _BL, _P = C.POINTER(Level), C.POINTER(Bloch), C.c_void_p
for _name, _args in (
        ("mxh_gram_cols", [_LV, _BL, C.c_int, _P, _P, C.c_int, Vecs, _P, _P, _P]),
        ("mxh_defect", [C.c_int, _LV, _BL, C.c_int, Vecs, Vecs, _P, _P, _P, _P]),
        ("mxh_lift_rhs", [C.c_int, _LV, _BL, C.c_int, Vecs, Vecs, Vecs, Vecs, Vecs, _P, _P]),
        ("mxh_lift_apply", [C.c_int, _LV, _BL, C.c_int, Vecs, Vecs, Vecs, Vecs, C.c_double, _P, _P]),
        ("mxh_lobpcg_combine", [C.c_longlong, C.c_int, _P, C.c_int, Vecs, Vecs, _P]),
        ("mxh_afw_march", [C.c_int, _LV, _BL, C.c_int, Vecs, Vecs, Vecs, _P, C.c_int, Vecs, Vecs, Vecs, C.c_int,
                           C.c_int]),
        ("mxh_gram_work_bytes", [C.c_int, C.c_int])):
    getattr(LIB, _name).argtypes = _args
LIB.mxh_gram_work_bytes.restype = C.c_size_t


def _vecs(t, stride):
    return Vecs(t.data_ptr() if t is not None else None, stride, None)


def _check(status):
    if status:
        raise RuntimeError("the library returned %d" % status)


class _View:
    """A device vector of the library as an array that torch can look at; keeps its owner alive."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n, 2), "typestr": "<f8", "data": (ptr, False), "version": 2}


def _tensor_of(edge):
    """The values of a module-API edge vector (struct: grid, x, y) as a tensor, without a copy."""
    ptr = C.cast(edge.h, C.POINTER(C.c_void_p))[1]
    return torch.view_as_complex(torch.as_tensor(_View(ptr, edge.n, edge), device="cuda"))


# ------------------------------------------------------------------ inputs from the seed
def _gen(seed, what=0):
    return torch.Generator(device=_dev()).manual_seed(1000003 * what + int(seed))


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _normal(gen, *shape, dtype=CD):
    """Complex Gaussian entries."""
    real = D if dtype == CD else torch.float32
    return torch.view_as_complex(torch.randn(*shape, 2, generator=gen, dtype=real, device=_dev()))


def _eta(pattern, nx, ny, seed):
    """1/eps per cell: rods in air whose radii and eps vary with the seed, or a two-phase random medium."""
    rng = np.random.default_rng(seed)
    if pattern == "medium":
        f = rng.standard_normal((ny, nx))
        ky, kx = np.fft.fftfreq(ny)[:, None], np.fft.fftfreq(nx)[None, :]
        s = max(2.0, 6.0 * nx / 256.0)
        f = np.real(np.fft.ifft2(np.fft.fft2(f) * np.exp(-2.0 * (np.pi * s) ** 2 * (kx ** 2 + ky ** 2))))
        return np.where(f > 0.0, 1.0 / 8.9, 1.0)
    X, Y = np.meshgrid(np.arange(nx) / nx, np.arange(ny) / ny)
    eta = np.ones((ny, nx))
    if pattern == "rod":
        rods = [(0.5, 0.5, 0.2 * rng.uniform(0.95, 1.05), 8.9 * rng.uniform(0.97, 1.03))]
    else:
        rods = [((a + 0.5) / 2, (b + 0.5) / 2, 0.5 * rng.uniform(0.15, 0.25), rng.uniform(6.0, 12.0))
                for b in range(2) for a in range(2)]
    for cx, cy, r, eps in rods:
        eta[(X - cx) ** 2 + (Y - cy) ** 2 <= r * r] = 1.0 / eps
    return eta


def _kpoints(case, seed):
    """A Gamma-X-M-Gamma path (both ends included from 8 points on), or neighbouring points of a Brillouin-zone grid."""
    count = case["problems"]
    if case["ks"] == "zone":
        k = -np.pi + 2.0 * np.pi * np.arange(32) / 31
        at = (seed * 64) % (1024 - count) + np.arange(count)
        return k[at % 32], k[at // 32]
    total = (2.0 + math.sqrt(2.0)) * math.pi
    s = np.arange(count) * total / (count - 1) if count >= 8 else (np.arange(count) + 0.5) * total / count
    kx = np.where(s <= np.pi, s, np.where(s <= 2 * np.pi, np.pi, np.maximum(np.pi - (s - 2 * np.pi) / math.sqrt(2.0), 0)))
    ky = np.where(s <= np.pi, 0.0, np.where(s <= 2 * np.pi, s - np.pi, kx))
    if count >= 8:
        kx[-1] = ky[-1] = 0.0
    return kx, ky


def _angles(seed, problems=1):
    rng = np.random.default_rng(seed + 77)
    return rng.uniform(0.4, 2.8, problems), rng.uniform(-2.8, -0.4, problems)


def _level(case):
    """A cell of one length unit in x; square meshes on square grids, others with hx != hy."""
    nx, ny = case["nx"], case["ny"]
    return Level(nx, ny, 1.0 / nx, 1.0 / ny)


def _block_inputs(case, seed):
    """What a block-step kernel reads, by name (device tensors; complex128 unless the case's precision is FP32)."""
    kind, nx, ny = case["kind"], case["nx"], case["ny"]
    N = nx * ny
    g = _gen(seed)
    problems = case.get("problems", 1)
    kx, ky = _angles(seed, problems)
    d = dict(kx=kx, ky=ky, eta=torch.from_numpy(_eta("rod", nx, ny, seed)).to(_dev()))
    low = torch.complex64 if case.get("prec") == F32 else CD
    if kind == "gram":
        d["u"] = _normal(g, problems, case["m"], 2 * N)
        rng = np.random.default_rng(seed)
        m, third = case["m"], case["m"] // 3
        cols = np.zeros((problems, m + 1), np.int32)
        for p in range(problems):  # the W columns (the middle third) of locked vectors are left out
            out = rng.choice(np.arange(third, 2 * third), m - case["cols"], replace=False) if case["cols"] < m else []
            cols[p, 0] = case["cols"]
            cols[p, 1:1 + case["cols"]] = np.setdiff1d(np.arange(m), out)
        d["cols"] = cols
    elif kind == "defect":
        d["e"] = _normal(g, case["nv"], 2 * N)
        d["lam"] = torch.linspace(1.2, 40.0, case["nv"], dtype=D, device=_dev())
    elif kind == "lift":
        d["e"] = _normal(g, case["nv"], 2 * N)
        d["x"] = 0.1 * _normal(g, case["nv"], 2 * N, dtype=low)
        d["xg"] = _normal(g, case["nv"], N, dtype=low)
    elif kind == "update":
        d["x"] = _normal(g, problems, 3 * case["m"], 2 * N)
        d["c"] = _normal(g, problems, 2 * case["m"], 3 * case["m"])  # column-major: [output, input]
    elif kind == "smooth":
        d["b"] = _normal(g, case["nv"], 2 * N)
        d["x"] = _normal(g, case["nv"], 2 * N)
        d["xc"] = _normal(g, case["nv"], N // 2)
    return d


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, seed)
    state["case"] = case
    torch.cuda.synchronize()
    return state


def run(state):
    return globals()["_run_" + state["case"]["kind"]](state)


def _solver(case, eta):
    return mx.Solver(eta, n0=case["n0"], levels=case["levels"], precision=case.get("prec", F64), block=case["block"],
                     max_problems=case.get("problems", 1), autotune=case.get("autotune", False),
                     method=mx.MX_METHOD_LOBPCG if case.get("method") == "lobpcg" else mx.MX_METHOD_PINVIT)


def _prepare_solve(case, seed):
    n = case["n0"] << case["levels"]
    kx, ky = _kpoints(case, seed)
    return dict(S=_solver(case, _eta(case["pattern"], n, n, seed)), kx=kx, ky=ky, seed=seed + 1)


def _run_solve(s):
    c = s["case"]
    r = s["S"].solve(s["kx"], s["ky"], c["neig"], tol=1e-8, maxit=400, seed=s["seed"])
    # the wanted eigenvalues; residuals and step counts are where the iteration
    # happened to stop below the tolerance, not a value it computes
    return r["lam"][:, :c["neig"]], r["converged"].astype(np.int64)


def _prepare_gradient(case, seed):
    n = case["n0"] << case["levels"]
    kx, ky = _angles(seed)
    S = _solver(case, _eta("medium", n, n, seed))
    S.solve(kx, ky, case["neig"], tol=1e-10, maxit=400, seed=seed + 1)
    return dict(S=S)


def _run_gradient(s):
    c = s["case"]
    return s["S"].eta_gradient(0, c["first"], c["count"])


def _prepare_block(case, seed):
    LIB.mxh_init()
    d = _block_inputs(case, seed)
    d["lv"] = _level(case)
    f = np.stack([np.cos(d["kx"]), np.sin(d["kx"]), np.cos(d["ky"]), np.sin(d["ky"])], 1)
    d["factors"] = torch.from_numpy(f).to("cuda")
    d["bl"] = Bloch(*f[0], d["factors"].data_ptr() if len(f) > 1 else None, case.get("m", 1), None)
    return d


def _prepare_gram(case, seed):
    d = _prepare_block(case, seed)
    m = case["m"]
    d["cols"] = torch.from_numpy(d["cols"]).to("cuda")
    d["out"] = torch.zeros(case["problems"], m * (m + 1) // 2, 4, dtype=D, device="cuda")
    d["work"] = torch.empty(LIB.mxh_gram_work_bytes(m, case["problems"]), dtype=torch.uint8, device="cuda")
    return d


def _run_gram(s):
    c, k = s["case"], s["case"]["cols"]
    n = 2 * c["nx"] * c["ny"]
    _check(LIB.mxh_gram_cols(C.byref(s["lv"]), C.byref(s["bl"]), c["problems"], None, s["cols"].data_ptr(), c["m"],
                             _vecs(s["u"], n), s["eta"].data_ptr(), s["out"].data_ptr(), s["work"].data_ptr()))
    return s["out"][:, :k * (k + 1) // 2]


def _prepare_defect(case, seed):
    d = _prepare_block(case, seed)
    nv, n = case["nv"], 2 * case["nx"] * case["ny"]
    d["r"] = torch.empty(nv, n, dtype=torch.complex64 if case["prec"] == F32 else CD, device="cuda")
    d["out"] = torch.empty(nv, 2, dtype=D, device="cuda")
    d["work"] = torch.empty(513 * 4 * nv + 1024, dtype=D, device="cuda")
    return d


def _run_defect(s):
    c, n = s["case"], 2 * s["case"]["nx"] * s["case"]["ny"]
    _check(LIB.mxh_defect(c["prec"], C.byref(s["lv"]), C.byref(s["bl"]), c["nv"], _vecs(s["e"], n), _vecs(s["r"], n),
                          s["eta"].data_ptr(), s["lam"].data_ptr(), s["out"].data_ptr(), s["work"].data_ptr()))
    return s["r"], s["out"]


def _prepare_lift(case, seed):
    d = _prepare_block(case, seed)
    nv, N = case["nv"], case["nx"] * case["ny"]
    d["bg"] = torch.empty(nv, N, dtype=d["xg"].dtype, device="cuda")
    d["coef"] = torch.empty(nv, 2, dtype=D, device="cuda")
    d["w"] = torch.empty(nv, 2 * N, dtype=CD, device="cuda")
    d["work"] = torch.empty(513 * 4 * nv + 1024, dtype=D, device="cuda")
    return d


def _run_lift(s):
    c, N = s["case"], s["case"]["nx"] * s["case"]["ny"]
    lv, bl, none = C.byref(s["lv"]), C.byref(s["bl"]), Vecs(None, 0, None)
    _check(LIB.mxh_lift_rhs(c["prec"], lv, bl, c["nv"], _vecs(s["e"], 2 * N), _vecs(s["x"], 2 * N), none,
                            _vecs(s["bg"], N), none, s["coef"].data_ptr(), s["work"].data_ptr()))
    _check(LIB.mxh_lift_apply(c["prec"], lv, bl, c["nv"], _vecs(s["xg"], N), none, _vecs(s["x"], 2 * N),
                              _vecs(s["w"], 2 * N), -1.0, s["coef"].data_ptr(), s["work"].data_ptr()))
    return s["bg"], s["coef"], s["w"]


def _prepare_update(case, seed):
    d = _prepare_block(case, seed)
    d["y"] = torch.zeros_like(d["x"])
    return d


def _run_update(s):
    c, m, n = s["case"], s["case"]["m"], 2 * s["case"]["nx"] * s["case"]["ny"]
    _check(LIB.mxh_lobpcg_combine(n, c["problems"], None, m, _vecs(s["x"], n), _vecs(s["y"], n), s["c"].data_ptr()))
    return s["y"][:, :m], s["y"][:, 2 * m:]


def _prepare_smooth(case, seed):
    d = _prepare_block(case, seed)
    d["down"], d["up"] = torch.empty_like(d["x"]), torch.empty_like(d["x"])
    d["bc"], d["xc0"] = torch.empty_like(d["xc"]), torch.empty_like(d["xc"])
    return d


def _run_smooth(s):
    c, N = s["case"], s["case"]["nx"] * s["case"]["ny"]
    lv, bl, none = C.byref(s["lv"]), C.byref(s["bl"]), Vecs(None, 0, None)
    b, eta = _vecs(s["b"], 2 * N), s["eta"].data_ptr()
    _check(LIB.mxh_afw_march(F64, lv, bl, c["nv"], b, _vecs(s["x"], 2 * N), _vecs(s["down"], 2 * N), eta, 8, none,
                             _vecs(s["bc"], N // 2), _vecs(s["xc0"], N // 2), 192, 2))
    _check(LIB.mxh_afw_march(F64, lv, bl, c["nv"], b, _vecs(s["down"], 2 * N), _vecs(s["up"], 2 * N), eta, 5,
                             _vecs(s["xc"], N // 2), none, none, 192, 2))
    return s["down"], s["bc"], s["up"]


def _random_fields(count, n, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal((count, n)) + 1j * r.standard_normal((count, n))


def _pointers(vectors):
    return (C.c_void_p * len(vectors))(*[v.h for v in vectors])


def _prepare_vector_step(case, seed):
    n, L = case["n0"] << case["levels"], case["levels"]
    kx, ky = _angles(seed)
    grids = [mx.Grid(_eta("rod", n, n, seed), kx[0], ky[0])]
    for _ in range(L):
        grids.insert(0, grids[0].coarse())
    e0 = _random_fields(1, 2 * n * n, seed)[0]
    s = dict(grids=grids, e0=mx.Edge(grids[L], e0), e=mx.Edge(grids[L], e0), lam=7.5)
    for name in "bxd":
        s[name] = [mx.Edge(g) for g in grids]
        s["n" + name] = [mx.Node(g) for g in grids]
    g0, n0 = grids[0], grids[0].nx * grids[0].ny
    s["Ae"], s["An"] = LIB.new_matrix(2 * n0, 2 * n0), LIB.new_matrix(n0, n0)
    LIB.densematrix_edge2d(mx.Cplx.of(1.0), mx.Cplx.of(1.0), g0.g, s["Ae"])
    LIB.densematrix_node2d(True, g0.g, s["An"])
    _check(LIB.potrf_matrix(s["Ae"]) or LIB.potrf_matrix(s["An"]))
    s["out"] = _tensor_of(s["e"])
    return s


def _run_vector_step(s):
    c = s["case"]
    LIB.copy_edge2d(s["e0"].h, s["e"].h)
    LIB.pinvit_edge2d(c["levels"], 2, c["prec_steps"], c["gradient_steps"], s["lam"], s["e"].h, s["Ae"],
                      _pointers(s["b"]), _pointers(s["x"]), _pointers(s["d"]), s["An"], _pointers(s["nb"]),
                      _pointers(s["nx"]), _pointers(s["nd"]))
    return s["out"]


def _prepare_ritz_rows(case, seed):
    nx, ny = case["nx"], case["ny"]
    kx, ky = _angles(seed)
    g = mx.Grid(_eta("rod", nx, ny, seed), kx[0], ky[0])
    return dict(grid=g, v=[mx.Edge(g, x) for x in _random_fields(case["vectors"], 2 * nx * ny, seed)])


def _run_ritz_rows(s):
    one, v, out = mx.Cplx.of(1.0), s["v"], []
    for a in range(len(v)):
        for b in range(a + 1):
            out.append(LIB.energyprod_edge2d(one, one, v[b].h, v[a].h).value())
            out.append(LIB.massprod_edge2d(v[b].h, v[a].h).value())
    return np.array(out).reshape(-1, 2)


def _prepare_orthonormalize(case, seed):
    nx, ny = case["nx"], case["ny"]
    kx, ky = _angles(seed)
    g = mx.Grid(_eta("rod", nx, ny, seed), kx[0], ky[0])
    v0 = [mx.Edge(g, x) for x in _random_fields(case["vectors"], 2 * nx * ny, seed)]
    v = [mx.Edge(g) for _ in v0]
    return dict(grid=g, v0=v0, v=v, work=mx.Edge(g), tau=(mx.Cplx * len(v))(), out=[_tensor_of(x) for x in v])


def _run_orthonormalize(s):
    for x, y in zip(s["v0"], s["v"]):
        LIB.copy_edge2d(x.h, y.h)
    LIB.orthonormalize_edge2d(len(s["v"]), _pointers(s["v"]), s["tau"], s["work"].h)
    return s["out"], np.array([t.value() for t in s["tau"]])


# ------------------------------------------------------------------ the work of one pass
def work(case):
    kind = case["kind"]
    n = case["n0"] << case["levels"] if "n0" in case else 0
    N = n * n if n else case["nx"] * case["ny"]
    E, eta = 2 * N, 8 * N
    if kind == "solve":
        # eta in, the block's vectors out and their Rayleigh-Ritz step once:
        # how many steps that takes is the method's affair
        nv = case["problems"] * case["block"]
        return dict(bytes=eta + 16 * E * nv, flops=N * case["problems"] * case["block"] * (case["block"] + 1) / 2 * 24)
    if kind == "gradient":
        return dict(bytes=2 * eta + 16 * E * case["count"], flops=40 * N * case["count"])
    if kind == "gram":
        k = case["cols"]
        return dict(bytes=eta + 16 * E * k * case["problems"], flops=24 * N * case["problems"] * k * (k + 1) / 2)
    low = 8 if case.get("prec") == F32 else 16
    if kind == "defect":
        return dict(bytes=eta + (16 + low) * E * case["nv"], flops=70 * N * case["nv"])
    if kind == "lift":
        # e, x and xg in; right-hand side and update out
        return dict(bytes=case["nv"] * (16 * E + low * E + low * N + low * N + 16 * E), flops=60 * N * case["nv"])
    if kind == "update":
        m = case["m"]
        return dict(bytes=5 * m * 16 * E * case["problems"], flops=8 * 3 * m * m * E * case["problems"])
    if kind == "smooth":
        # b, x, xc in; x after the way down, the coarse right-hand side and x after the way up out
        return dict(bytes=eta + case["nv"] * 16 * (2 * E + E / 4 + E + E / 4 + E), flops=4 * 180 * N * case["nv"])
    if kind == "vector_step":
        # e in and out, eta in; four edge sweeps a cycle over all levels (4/3), four nodal ones
        flops = 4 / 3 * N * (case["prec_steps"] * 4 * 180 + case["gradient_steps"] * 4 * 30)
        return dict(bytes=eta + 32 * E, flops=flops)
    k = case["vectors"]
    if kind == "ritz_rows":
        return dict(bytes=eta + 16 * E * k, flops=k * (k + 1) / 2 * 2 * 100 * N)
    return dict(bytes=2 * 16 * E * k, flops=2 * 16 * E * k * k)


# ------------------------------------------------------------------ the same in plain torch, 64 bits
class _Ref:
    """Operators of a periodic Bloch grid on arrays (..., ny, nx)."""

    def __init__(self, eta, hx, hy, kx, ky):
        self.eta, self.hx, self.hy = eta.to(CD), hx, hy
        self.kx, self.ky = kx, ky
        self.ny, self.nx = eta.shape
        self.mx, self.my, self.s = hy / hx / 6.0, hx / hy / 6.0, 1.0 / (hx * hy)

    def at(self, a, di, dj, phase=True):
        """a(i + di, j + dj) through the Bloch relation."""
        b = torch.roll(a, (-dj, -di), (-2, -1))
        if not phase:
            return b
        i = torch.arange(self.nx, device=a.device) + di
        j = torch.arange(self.ny, device=a.device) + dj
        over = [(k >= n).to(D) - (k < 0).to(D) for k, n in ((i, self.nx), (j, self.ny))]
        ph = self.kx * over[0] + self.ky * over[1][:, None]
        return b * torch.polar(torch.ones_like(ph), ph)

    def split(self, v):
        v = v.reshape(*v.shape[:-1], 2, self.ny, self.nx)
        return v[..., 0, :, :], v[..., 1, :, :]

    def join(self, x, y):
        return torch.stack((x, y), -3).reshape(*x.shape[:-2], -1)

    def curl(self, x, y):
        return x - self.at(x, 0, 1) - y + self.at(y, 1, 0)

    def mass(self, x, y):
        return (self.mx * (4 * x + self.at(x, 0, 1) + self.at(x, 0, -1)),
                self.my * (4 * y + self.at(y, 1, 0) + self.at(y, -1, 0)))

    def apply(self, x, y, beta=1.0):
        q = self.s * self.eta * self.curl(x, y)
        a, b = self.mass(x, y)
        return q - self.at(q, 0, -1) + beta * a, self.at(q, -1, 0) - q + beta * b

    def colour(self, ci, cj):
        m = torch.zeros(self.ny, self.nx, dtype=torch.bool, device=self.eta.device)
        m[cj::2, ci::2] = True
        return m

    def afw(self, bx, by, x, y, backward=False):
        """One four-colour sweep of exact vertex-patch solves (doubled mass diagonal)."""
        e = self.s * self.eta
        ll, rl, lu, ru = (self.at(e, di, dj, False) for di, dj in ((-1, -1), (0, -1), (-1, 0), (0, 0)))
        a0, a1 = ll + lu + 8 * self.mx, rl + ru + 8 * self.mx
        a2, a3 = ll + rl + 8 * self.my, lu + ru + 8 * self.my
        s22, s33 = a2 - ll * ll / a0 - rl * rl / a1, a3 - lu * lu / a0 - ru * ru / a1
        s23 = ll * lu / a0 + rl * ru / a1
        det = s22 * s33 - s23 * s23
        for c in range(3, -1, -1) if backward else range(4):
            ax, ay = self.apply(x, y)
            r1, r3 = bx - ax, by - ay
            r0, r2 = self.at(r1, -1, 0), self.at(r3, 0, -1)
            t2 = r2 + ll / a0 * r0 - rl / a1 * r1
            t3 = r3 - lu / a0 * r0 + ru / a1 * r1
            z2, z3 = (s33 * t2 - s23 * t3) / det, (s22 * t3 - s23 * t2) / det
            z0 = (r0 + ll * z2 - lu * z3) / a0
            z1 = (r1 - rl * z2 + ru * z3) / a1
            m = self.colour(c & 1, c >> 1)
            z0, z1, z2, z3 = (z * m for z in (z0, z1, z2, z3))
            x = x + z1 + self.at(z0, 1, 0)
            y = y + z3 + self.at(z2, 0, 1)
        return x, y

    def restrict(self, x, y):
        a = 0.5 * x + 0.25 * (self.at(x, 0, 1) + self.at(x, 0, -1))
        b = 0.5 * y + 0.25 * (self.at(y, 1, 0) + self.at(y, -1, 0))
        return ((a + self.at(a, 1, 0))[..., ::2, ::2], (b + self.at(b, 0, 1))[..., ::2, ::2])

    def prolong(self, coarse, x, y):
        fx = torch.zeros(*x.shape[:-2], self.ny, self.nx, dtype=CD, device=x.device)
        fy = torch.zeros_like(fx)
        fx[..., ::2, ::2] = fx[..., ::2, 1::2] = 0.5 * x
        fx[..., 1::2, ::2] = fx[..., 1::2, 1::2] = 0.25 * (x + coarse.at(x, 0, 1))
        fy[..., ::2, ::2] = fy[..., 1::2, ::2] = 0.5 * y
        fy[..., ::2, 1::2] = fy[..., 1::2, 1::2] = 0.25 * (y + coarse.at(y, 1, 0))
        return fx, fy

    def node(self, v):
        """The Q1 Laplacian (stiffness in one direction, mass in the other)."""
        h, k = self.hx, self.hy
        tx = self.at(v, 1, 0) + self.at(v, -1, 0)
        ty = self.at(v, 0, 1) + self.at(v, 0, -1)
        txy = self.at(tx, 0, 1) + self.at(tx, 0, -1)
        return (4 * (h / k + k / h) / 3 * v + (h / k - 2 * k / h) / 3 * tx + (k / h - 2 * h / k) / 3 * ty -
                (h / k + k / h) / 6 * txy)

    def node_sweep(self, b, v, backward=False):
        d = 4 * (self.hx / self.hy + self.hy / self.hx) / 3
        for c in range(3, -1, -1) if backward else range(4):
            v = v + (b - self.node(v)) / d * self.colour(c & 1, c >> 1)
        return v

    def node_restrict(self, r):
        t = r + 0.5 * (self.at(r, 1, 0) + self.at(r, -1, 0))
        return (t + 0.5 * (self.at(t, 0, 1) + self.at(t, 0, -1)))[..., ::2, ::2]

    def node_prolong(self, coarse, v):
        f = torch.zeros(*v.shape[:-2], self.ny, self.nx, dtype=CD, device=v.device)
        vx, vy = coarse.at(v, 1, 0), coarse.at(v, 0, 1)
        f[..., ::2, ::2] = v
        f[..., ::2, 1::2] = 0.5 * (v + vx)
        f[..., 1::2, ::2] = 0.5 * (v + vy)
        f[..., 1::2, 1::2] = 0.25 * (v + vx + vy + coarse.at(vx, 0, 1))
        return f

    def gradient(self, v):
        return self.at(v, 1, 0) - v, self.at(v, 0, 1) - v

    def adjgradient(self, x, y):
        return self.at(x, -1, 0) - x + self.at(y, 0, -1) - y

    def wave(self):
        """The lowest Bloch plane wave of the node space and its Laplacian eigenvalue."""
        tx, ty = self.kx / self.nx, self.ky / self.ny
        i = torch.arange(self.nx, device=self.eta.device, dtype=D)
        j = torch.arange(self.ny, device=self.eta.device, dtype=D)
        ph = tx * i + ty * j[:, None]
        sx, sy = 2 * math.sin(tx / 2) ** 2, 2 * math.sin(ty / 2) ** 2
        rx, ry = self.hy / self.hx, self.hx / self.hy
        mu = rx * 2 * sx * (1 - sy / 3) + ry * 2 * sy * (1 - sx / 3)
        return torch.polar(torch.ones_like(ph), ph), mu


def exact(case, seed):
    f = globals()["_exact_" + case["kind"]]
    return f(case, seed)


def _ref(case, seed, d, p=0):
    return _Ref(d["eta"], 1.0 / case["nx"], 1.0 / case["ny"], float(d["kx"][p]), float(d["ky"][p]))


def _orth(Q):
    """Orthonormal columns by two passes of Cholesky QR."""
    for _ in range(2):
        R = torch.linalg.cholesky(Q.mH @ Q, upper=True)
        Q = torch.linalg.solve_triangular(R, Q, upper=True, left=False)
    return Q


def _bands(eta, kx, ky, count):
    """The smallest `count` nonzero eigenvalues of the curl-curl pencil and their fields f = sqrt(eta) curl u.

    K = C^H eta C / (hx hy) and M is diagonal in the twisted Fourier basis, so the nonzero spectrum is that of
    sqrt(eta) S sqrt(eta) on the cells with S = C M^-1 C^H / (hx hy), whose inverse is one FFT pair between two
    diagonal scalings: block Krylov steps with the inverse find its lowest end to rounding."""
    ny, nx = eta.shape
    dev = eta.device
    i, j = torch.arange(nx, device=dev, dtype=D), torch.arange(ny, device=dev, dtype=D)
    tx = (2 * math.pi * torch.fft.fftfreq(nx, device=dev, dtype=D) + kx / nx)[None, :]
    ty = (2 * math.pi * torch.fft.fftfreq(ny, device=dev, dtype=D) + ky / ny)[:, None]
    hx, hy = 1.0 / nx, 1.0 / ny
    S = (4 * torch.sin(ty / 2) ** 2 / (hy / hx / 6 * (4 + 2 * torch.cos(ty))) +
         4 * torch.sin(tx / 2) ** 2 / (hx / hy / 6 * (4 + 2 * torch.cos(tx)))) / (hx * hy)
    gamma = kx == 0.0 and ky == 0.0
    inv = torch.where(S > 1e-12 * S.max(), 1.0 / S, torch.zeros_like(S)) if gamma else 1.0 / S
    twist = torch.polar(torch.ones(ny, nx, dtype=D, device=dev), kx / nx * i + ky / ny * j[:, None])
    root = torch.sqrt(1.0 / eta)  # sqrt(eps)
    null = (root / root.norm()).reshape(-1, 1).to(CD)

    def op(F):  # columns
        if gamma:
            F = F - null @ (null.mH @ F)
        G = F.T.reshape(-1, ny, nx) * (root * twist.conj())
        G = torch.fft.ifft2(torch.fft.fft2(G) * inv) * (root * twist)
        G = G.reshape(-1, ny * nx).T
        return G - null @ (null.mH @ G) if gamma else G

    width = count + 6
    gen = torch.Generator(device=dev).manual_seed(3)
    X = _orth(op(op(torch.view_as_complex(torch.randn(ny * nx, width, 2, generator=gen, dtype=D, device=dev)))))
    for _ in range(12):  # restarted Krylov spaces of three blocks
        blocks = [X]
        for _ in range(2):
            B = op(blocks[-1])
            for _ in range(2):
                for Q in blocks:
                    B = B - Q @ (Q.mH @ B)
            blocks.append(_orth(B))
        V = torch.cat(blocks, 1)
        T = V.mH @ op(V)
        w, U = torch.linalg.eigh(((T + T.mH) / 2).cpu())
        X = V @ U[:, -width:].flip(1).to(dev)
        w = w.flip(0)[:count]
        if gamma:
            X = X - null @ (null.mH @ X)
        X = _orth(X)
        rest = (op(X[:, :count]) - X[:, :count] * w.to(dev)).norm(dim=0)
        if float((rest / w.to(dev)).max()) < 1e-10:
            break
    return 1.0 / w, X[:, :count]


def _exact_solve(case, seed):
    n = case["n0"] << case["levels"]
    if n * n * case["problems"] > 64 * 256 * 256:
        return None
    eta = torch.from_numpy(_eta(case["pattern"], n, n, seed)).to(_dev())
    kx, ky = _kpoints(case, seed)
    lam = [_bands(eta, float(a), float(b), case["neig"])[0].numpy() for a, b in zip(kx, ky)]
    return np.stack(lam), None


def _exact_gradient(case, seed):
    n = case["n0"] << case["levels"]
    eta = torch.from_numpy(_eta("medium", n, n, seed)).to(_dev())
    kx, ky = _angles(seed)
    lam, F = _bands(eta, float(kx[0]), float(ky[0]), 6)
    at = slice(case["first"], case["first"] + case["count"])
    F = F[:, at]
    g = (F.abs() ** 2 / F.norm(dim=0) ** 2 * lam[at].to(F.device)).sum(1).reshape(n, n) / eta
    return g.cpu().numpy()


def _exact_gram(case, seed):
    d, k, out = _block_inputs(case, seed), case["cols"], []
    rows, cols = np.tril_indices(k)
    for p in range(case["problems"]):
        r = _ref(case, seed, d, p)
        u = d["u"][p][torch.from_numpy(d["cols"][p, 1:1 + k].astype(np.int64)).to(d["u"].device)]
        x, y = r.split(u)
        c = r.curl(x, y).reshape(k, -1)
        gk = c.conj() @ (c * r.eta.reshape(-1)).T
        gm = u.conj() @ r.join(*r.mass(x, y)).T
        g = torch.stack((gk.real, gk.imag, gm.real, gm.imag), -1)
        out.append(g[rows, cols])
    return torch.stack(out)


def _exact_defect(case, seed):
    d = _block_inputs(case, seed)
    r, rs, norms = _ref(case, seed, d), [], []
    for e, lam in zip(d["e"], d["lam"].tolist()):
        x, y = r.split(e)
        v, m = r.join(*r.apply(x, y, 1.0 - lam)), r.join(*r.mass(x, y))
        rs.append(v)
        norms.append(torch.stack((v.abs().square().sum(), m.abs().square().sum())))
    return torch.stack(rs), torch.stack(norms)


def _exact_lift(case, seed):
    d = _block_inputs(case, seed)
    r, N = _ref(case, seed, d), case["nx"] * case["ny"]
    phi, mu = r.wave()
    bgs, coefs, ws = [], [], []
    for e, x, xg in zip(d["e"], d["x"].to(CD), d["xg"].to(CD)):
        b = r.adjgradient(*r.mass(*r.split(e - x)))
        c = (phi.conj() * b).sum() / N
        bgs.append((b - c * phi).reshape(-1))
        coefs.append(torch.view_as_real(c / mu))
        v = xg.reshape(case["ny"], case["nx"])
        v = v + (c / mu - (phi.conj() * v).sum() / N) * phi
        ws.append(-x - r.join(*r.gradient(v)))
    return torch.stack(bgs), torch.stack(coefs), torch.stack(ws)


def _exact_update(case, seed):
    d, m = _block_inputs(case, seed), case["m"]
    E, P = [], []
    for x, c in zip(d["x"], d["c"]):
        c = c[:m]
        P.append(c[:, m:] @ x[m:])
        E.append(c[:, :m] @ x[:m] + P[-1])
    return torch.stack(E), torch.stack(P)


def _exact_smooth(case, seed):
    d = _block_inputs(case, seed)
    r = _ref(case, seed, d)
    coarse = _Ref(d["eta"][::2, ::2], 2 * r.hx, 2 * r.hy, r.kx, r.ky)
    downs, bcs, ups = [], [], []
    for b, x0, xc in zip(d["b"], d["x"], d["xc"]):
        bx, by = r.split(b)
        x, y = r.split(x0)
        for _ in range(2):
            x, y = r.afw(bx, by, x, y)
        ax, ay = r.apply(x, y)
        downs.append(r.join(x, y))
        bcs.append(coarse.join(*r.restrict(bx - ax, by - ay)))
        px, py = r.prolong(coarse, *coarse.split(xc))
        x, y = x + px, y + py
        for _ in range(2):
            x, y = r.afw(bx, by, x, y, True)
        ups.append(r.join(x, y))
    return torch.stack(downs), torch.stack(bcs), torch.stack(ups)


def _exact_vector_step(case, seed):
    n, L = case["n0"] << case["levels"], case["levels"]
    kx, ky = (float(k[0]) for k in _angles(seed))
    eta = torch.from_numpy(_eta("rod", n, n, seed)).to(_dev())
    refs = [_Ref(eta, 1.0 / n, 1.0 / n, kx, ky)]
    for _ in range(L):
        eta = 0.25 * (eta[::2, ::2] + eta[::2, 1::2] + eta[1::2, ::2] + eta[1::2, 1::2])
        refs.insert(0, _Ref(eta, 2 * refs[0].hx, 2 * refs[0].hy, kx, ky))
    c, n0 = refs[0], case["n0"] ** 2
    Ae = c.join(*c.apply(*c.split(torch.eye(2 * n0, dtype=CD, device=_dev())))).T
    An = c.node(torch.eye(n0, dtype=CD, device=_dev()).reshape(n0, c.ny, c.nx)).reshape(n0, n0).T

    def edge_cycle(l, bx, by, x, y):
        r = refs[l]
        if l == 0:
            return r.split(torch.linalg.solve(Ae, r.join(bx, by)))
        for _ in range(2):
            x, y = r.afw(bx, by, x, y)
        ax, ay = r.apply(x, y)
        rx, ry = r.restrict(bx - ax, by - ay)
        cx, cy = edge_cycle(l - 1, rx, ry, torch.zeros_like(rx), torch.zeros_like(ry))
        px, py = r.prolong(refs[l - 1], cx, cy)
        x, y = x + px, y + py
        for _ in range(2):
            x, y = r.afw(bx, by, x, y, True)
        return x, y

    def node_cycle(l, b, v):
        r = refs[l]
        if l == 0:
            return torch.linalg.solve(An, b.reshape(-1)).reshape(r.ny, r.nx)
        for _ in range(2):
            v = r.node_sweep(b, v)
        bc = r.node_restrict(b - r.node(v))
        v = v + r.node_prolong(refs[l - 1], node_cycle(l - 1, bc, torch.zeros_like(bc)))
        for _ in range(2):
            v = r.node_sweep(b, v, True)
        return v

    r = refs[L]
    e = r.split(torch.from_numpy(_random_fields(1, 2 * n * n, seed)[0]).to(_dev()))
    bx, by = r.apply(*e, 1.0 - 7.5)
    x, y = torch.zeros_like(bx), torch.zeros_like(by)
    for _ in range(case["prec_steps"]):
        x, y = edge_cycle(L, bx, by, x, y)
    ux, uy = e[0] - x, e[1] - y
    b = r.adjgradient(*r.mass(ux, uy))
    v = torch.zeros_like(b)
    for _ in range(case["gradient_steps"]):
        v = node_cycle(L, b, v)
    gx, gy = r.gradient(v)
    return r.join(ux - gx, uy - gy)


def _module_ref(case, seed):
    nx, ny = case["nx"], case["ny"]
    kx, ky = (float(k[0]) for k in _angles(seed))
    eta = torch.from_numpy(_eta("rod", nx, ny, seed)).to(_dev())
    v = torch.from_numpy(_random_fields(case["vectors"], 2 * nx * ny, seed)).to(_dev())
    return _Ref(eta, 1.0 / nx, 1.0 / ny, kx, ky), v


def _exact_ritz_rows(case, seed):
    r, v = _module_ref(case, seed)
    x, y = r.split(v)
    a, m = r.join(*r.apply(x, y)), r.join(*r.mass(x, y))
    out = []
    for p in range(len(v)):
        for q in range(p + 1):
            out.append([torch.vdot(a[q], v[p]), torch.vdot(m[q], v[p])])
    return torch.tensor([[complex(e) for e in pair] for pair in out], dtype=CD).numpy()


def _exact_orthonormalize(case, seed):
    r, X = _module_ref(case, seed)
    k, nx, ny = len(X), r.nx, r.ny

    def mass(v):
        return r.join(*r.mass(*r.split(v)))

    units = torch.zeros_like(X)
    for i in range(k):
        units[i, i % nx + (1 + 2 * (i // nx)) * nx] = math.sqrt(0.25 / r.mx)
    Mu, tau = mass(units), []
    for i in range(k):
        alpha = math.sqrt(torch.vdot(X[i], mass(X[i])).real)
        beta = complex(torch.vdot(Mu[i], X[i]))
        alpha = -alpha if beta.real < 0 else alpha
        X[i] += alpha * units[i]
        tau.append(1.0 / (alpha * alpha + beta * alpha))
        if i + 1 < k:
            X[i + 1:] -= tau[i] * torch.outer(X[i + 1:] @ mass(X[i]).conj(), X[i])
            X[i + 1:] -= torch.outer(X[i + 1:] @ Mu[i].conj(), units[i])
    V = units.clone()
    for j in range(k - 1, -1, -1):
        V[j:] -= np.conj(tau[j]) * torch.outer(V[j:] @ mass(X[j]).conj(), X[j])
    return list(V), np.array(tau)
