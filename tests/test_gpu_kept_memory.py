"""An allocation that fails while the context keeps unused blocks gives them back
and is tried again, wherever a call allocates device memory.  The failure is the
host's: a library loaded before libmfdfd answers the n-th allocation of a call
with "out of memory"."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

pytestmark = pytest.mark.gpu

SHIM = """
#include <stddef.h>
int (*real)(void **, size_t) = 0;
int calls = 0, fail_at = -1;
int hipMalloc(void **p, size_t n) {
    if (calls++ == fail_at) { *p = 0; return 2; }   /* hipErrorOutOfMemory */
    return real(p, n);
}
"""

PROGRAM = """
import ctypes as C, os, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for p in ("maxwellfdm.jl_amd", "tests"):
    sys.path.insert(0, os.path.join(sys.argv[2], p))
import numpy as np
import maxwellfdfd as pkg
from test_gpu_resident import OM, TOL, system
pkg.lib()
hip = [l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l][0]
real = C.CDLL(hip).hipMalloc
C.c_void_p.in_dll(shim, "real").value = C.cast(real, C.c_void_p).value
calls, fail_at = C.c_int.in_dll(shim, "calls"), C.c_int.in_dll(shim, "fail_at")
m, rng = system(pkg, (9, 8, 7), (False,) * 3, (0, 0, 1), "diag", 71)
op = pkg.MaxwellOperator(m, OM)
x = rng.normal(size=op.n) + 0j
y = op.apply(x)
Acsc = pkg.to_scipy(pkg.A_csc(m, OM, m.εarr, m.μarr))
def small_batch():
    ops = [pkg.MaxwellOperator(m, OM) for _ in range(2)]
    es, _ = pkg.solve_batch(ops, [x, x], tol=TOL)
    for o in ops: o.close()
    return es[0]
def from_csc():
    o = pkg.MaxwellOperator.from_csc(Acsc)
    z = o.apply(x)
    o.close()
    return z
def materials():
    mm = pkg.ModelFull(pkg.Grid([np.arange(7.0)] * 3))
    pkg.add_obj(mm, "vacuum", pkg.Cuboid((3.0,) * 3, (6.0,) * 3), ε=1.0)
    pkg.add_obj(mm, "ball", pkg.Ball((3.0,) * 3, 2.0), ε=4.0)
    pkg.calc_matparams(mm)
    return mm.εarr
todo = dict(batch=small_batch, from_csc=from_csc, materials=materials, dls=lambda: pkg.create_stretched_dls(m),
            bench=lambda: (op.bench_apply(2, iters=1), 0)[1], assemble=lambda: pkg.A_csc(m, OM, m.εarr, m.μarr))
flat = lambda v: np.concatenate([flat(a) for a in v]) if isinstance(v, (list, tuple)) else np.asarray(v, complex).ravel()
for name, f in todo.items():
    calls.value = 0
    want = flat(f())
    n = calls.value
    print(name, n, "allocations", flush=True)
    for k in range(n + 1):
        op.apply(x)               # blocks are kept again
        calls.value, fail_at.value = 0, k
        got = flat(f())
        fail_at.value = -1
        assert np.array_equal(got, want), (name, k)
print("all ok", flush=True)
"""


def test_given_back(tmp_path):
    c, so, py = tmp_path / "few.c", tmp_path / "libfew.so", tmp_path / "program.py"
    c.write_text(SHIM)
    py.write_text(PROGRAM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(c)], check=True)
    p = subprocess.run([sys.executable, "-u", str(py), str(so), ROOT], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONDONTWRITEBYTECODE="1"))
    print(p.stdout)
    assert p.returncode == 0 and "all ok" in p.stdout, p.stdout + p.stderr
