"""What creating a solver allocates, counted on the CPU: the solver's C code with a
device that is host memory.  Pinning host memory costs about 25 us however little
is pinned, so a solver pins once."""
import ctypes as C
import os
import shutil
import subprocess

import numpy as np
import pytest

import maxwell_amd as M

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DEVICE = r"""
#include <stdlib.h>
#include <string.h>
#include "mxh.h"
int pinned, pinned_live, live, fail_pin;
int mxh_init(void) { return 0; }
int mxh_sync(void) { return 0; }
void *mxh_malloc(size_t n) { live++; return malloc(n); }
void mxh_free(void *p) { live -= !!p; free(p); }
void *mxh_host_alloc(size_t n) { if (fail_pin) return NULL; pinned++; pinned_live++; return malloc(n); }
void mxh_host_free(void *p) { pinned_live -= !!p; free(p); }
int mxh_h2d(void *d, const void *s, size_t n) { memcpy(d, s, n); return 0; }
int mxh_event_create(void **e) { *e = malloc(1); return 0; }
int mxh_event_destroy(void *e) { free(e); return 0; }
void mxh_graph_destroy(void *g) { (void)g; }
int mxh_cycle_supported(int prec, const mxh_cycle *c) { (void)prec; (void)c; return 0; }
int mxh_lift_supported(int prec, const mxh_level *l) { (void)prec; (void)l; return 0; }
size_t mxh_gram_work_bytes(int m, int nprob) { return (size_t)m * nprob; }
"""


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    if not shutil.which("gcc") or not shutil.which("nm"):
        pytest.skip("no compiler")
    d = tmp_path_factory.mktemp("host")
    inc = ["-I" + os.path.join(ROOT, "include")]
    src = os.path.join(ROOT, "maxwell_amd", "csrc", "bloch_solver.c")
    obj = str(d / "solver.o")
    subprocess.run(["gcc", "-std=gnu11", "-O1", "-fPIC", *inc, "-c", src, "-o", obj], check=True)
    # what the solver calls beyond creation ends the process here
    names = subprocess.run(["nm", "-u", obj], check=True, capture_output=True, text=True).stdout.split()
    rest = [n for n in names if n.startswith("mx") and " %s(" % n not in DEVICE.replace("*", " ")]
    (d / "device.c").write_text(DEVICE)
    (d / "rest.c").write_text("#include <stdlib.h>\n" + "".join("void %s(void) { abort(); }\n" % n for n in rest))
    so = str(d / "host.so")
    subprocess.run(["gcc", "-std=gnu11", "-fPIC", "-shared", *inc, str(d / "device.c"), str(d / "rest.c"), obj, "-o",
                    so, "-lm"], check=True)
    return C.CDLL(so)


def counter(host, name):
    return C.c_int.in_dll(host, name)


def create(host, method, block, problems):
    cfg = M.MxConfig(4, 2, M.MX_PREC_F64, block, problems, 2, 2, 5, 0, 1, 256, 192, 1, 0, 0, method)
    eta, h = np.ones((16, 16)), C.c_void_p()
    rc = host.mx_solver_create(C.byref(cfg), eta.ctypes.data_as(C.c_void_p), C.byref(h))
    return rc, h


@pytest.mark.parametrize("method", [M.MX_METHOD_PINVIT, M.MX_METHOD_LOBPCG])
@pytest.mark.parametrize("block,problems", [(1, 1), (3, 5), (16, 1)])
def test_one_pinned_allocation(host, method, block, problems):
    counter(host, "pinned").value = 0
    rc, h = create(host, method, block, problems)
    assert rc == 0 and counter(host, "pinned").value == 1
    host.mx_solver_destroy(h)
    assert counter(host, "pinned_live").value == 0 and counter(host, "live").value == 0


@pytest.mark.parametrize("method", [M.MX_METHOD_PINVIT, M.MX_METHOD_LOBPCG])
def test_no_pinned_memory_is_an_error(host, method):
    """MX_ENOMEM, and nothing kept."""
    counter(host, "fail_pin").value = 1
    rc, _ = create(host, method, 3, 2)
    counter(host, "fail_pin").value = 0
    assert rc == 2 and counter(host, "live").value == 0
