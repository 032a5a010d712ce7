"""xg_lu_solve_noalloc makes no allocating call: in a process of its own, a small
library ahead of the HIP runtime counts the allocations and graph
instantiations that libxyce_amd.so asks for."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#define _GNU_SOURCE
#include <dlfcn.h>
int counting = 0, calls = 0;
#define FORWARD(name)                                                                        \
  int name(long a, long b, long c, long d, long e, long f) {                                 \
    static int (*real)(long, long, long, long, long, long);                                  \
    if (!real) real = dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD), #name);     \
    calls += counting;                                                                       \
    return real(a, b, c, d, e, f);                                                           \
  }
FORWARD(hipMalloc) FORWARD(hipMallocAsync) FORWARD(hipHostMalloc) FORWARD(hipStreamCreate)
FORWARD(hipStreamBeginCapture) FORWARD(hipGraphInstantiate)
"""

CHILD = r"""
import ctypes, os, sys
sys.path.insert(0, os.getcwd())
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
counting, calls = (ctypes.c_int.in_dll(shim, k) for k in ("counting", "calls"))
import numpy as np
import xyce_amd as X
from xyce_amd import circuits as C
L = X.lib()
hip = ctypes.CDLL("libamdhip64.so.7")
V = ctypes.c_void_p

def device(a):
    p = V()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(a.nbytes)) == 0
    assert hip.hipMemcpy(p, a.ctypes.data_as(V), ctypes.c_size_t(a.nbytes), 1) == 0
    return p

def check(tag, n, rp, ci, values, method):
    counting.value, calls.value = 1, 0
    s = X.DirectSolver(n, rp, ci, method=method)
    assert calls.value > 0                     # the counter sees this library's calls
    b = np.random.default_rng(1).normal(size=n)
    bd, xd = device(b), device(np.zeros(n))
    for v in values:
        assert s.numeric(v) == 0
        for _ in range(2):
            calls.value = 0
            assert L.xg_lu_solve_noalloc(s.h, bd, xd) == 0
            print(tag, "allocating calls:", calls.value, flush=True)
            assert calls.value == 0
    counting.value = 0

def circuit(ckt):
    h = X.host_pattern(ckt)
    n, rp, ci = h["n"], h["rowptr"], h["colind"]
    v = np.where(ci == np.repeat(np.arange(n), np.diff(rp)), 9.0, -1.0)
    return n, rp, ci, (v, 2.0 * v)

def chain(n):                                  # zeros on the diagonal later: new pivots, a new plan
    rp = np.concatenate([[0], np.cumsum(np.where((np.arange(n) % (n - 1)) == 0, 2, 3))]).astype(np.int32)
    row = np.repeat(np.arange(n), np.diff(rp))
    ci = (row + np.concatenate([[0, 1], np.tile([-1, 0, 1], n - 2), [-1, 0]])).astype(np.int32)
    v = np.where(ci == row, 4.0, np.where(ci < row, -1.0, 1.0))
    return n, rp, ci, (v, np.where((ci == row) & (row % 7 == 3), 0.0, v))

check("ring 103", *circuit(C.ring(101)), 0)
check("ring 133", *circuit(C.ring(131)), 0)
check("gates 300", *circuit(C.gate_dag(300, seed=4)), 0)
check("grid 48 x 48", *circuit(C.power_grid(48, 48, seed=3, pad_pitch=16, n_sinks=32)), 2)
check("chain 400, new pivots", *chain(400), 0)
"""


def test_noalloc_solve_allocates_nothing(gpu, tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-w", "-o", str(so), str(src), "-ldl"], check=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CHILD, str(so)], cwd=root, capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr)
    assert r.returncode == 0
