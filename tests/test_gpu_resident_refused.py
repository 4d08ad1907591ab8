"""A device that refuses the resident solver's cooperative launch: the solve goes
on step by step.  In test_refused the refusal is the host's: a library loaded before libmfdfd
answers the launch with the runtime's error and starts nothing."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT
from test_gpu_resident import OM, TOL, system

pytestmark = pytest.mark.gpu

SHIM = """
int calls = 0;
int hipLaunchCooperativeKernel(const void *f, ...) { (void)f; ++calls; return ERROR; }
"""

PROGRAM = """
import ctypes as C, os, sys, time
start = time.monotonic()
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
for p in ("maxwellfdm.jl_amd", "oracle", "tests"):
    sys.path.insert(0, os.path.join(sys.argv[2], p))
import numpy as np
import maxwellfdfd as pkg, oracle as O
from conftest import spec_of
from test_gpu_resident import OM, TOL, system
made = []
for N in ((13, 9, 11), (10, 12, 7)):
    m, rng = system(pkg, N, (False,) * 3, (0, 0, 0), "diag", 51)
    made.append((pkg.MaxwellOperator(m, OM), O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)), rng))
def check(A, b, e):
    assert np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
def asked():   # once, and again after 10 s only
    n = C.c_int.in_dll(shim, "calls").value
    return 1 <= n <= 1 + (time.monotonic() - start) / 10
op, A, rng = made[0]
for precision in ("fp64", "mixed"):
    b = rng.normal(size=(2, A.shape[0])) + 1j * rng.normal(size=(2, A.shape[0]))
    for rhs in (b[0], b):
        e, st = op.solve(rhs, tol=TOL, precision=precision)
        for r, x in zip(np.atleast_2d(rhs), np.atleast_2d(e)):
            check(A, r, x)
print("single ok", flush=True)
assert asked()
op.close()
m, rng = system(pkg, (13, 9, 11), (False,) * 3, (0, 0, 0), "diag", 51)
made[0] = (pkg.MaxwellOperator(m, OM), A, rng)
bs = [rng.normal(size=A.shape[0]) + 0j for _, A, rng in made]
es, _ = pkg.solve_batch([op for op, _, _ in made], bs, tol=TOL)
for (_, A, _), b, e in zip(made, bs, es):
    check(A, b, e)
assert asked()
print("batch ok", flush=True)
"""


# hipErrorCooperativeLaunchTooLarge, hipErrorIllegalState, hipErrorNotSupported
@pytest.mark.parametrize("error", [720, 401, 801])
def test_refused(error, tmp_path):
    c, so, py = tmp_path / "refuse.c", tmp_path / "librefuse.so", tmp_path / "program.py"
    c.write_text(SHIM)
    py.write_text(PROGRAM)
    subprocess.run(["gcc", "-shared", "-fPIC", f"-DERROR={error}", "-o", str(so), str(c)], check=True)
    p = subprocess.run([sys.executable, "-u", str(py), str(so), ROOT], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONDONTWRITEBYTECODE="1"))
    assert p.returncode == 0 and "batch ok" in p.stdout, p.stdout + p.stderr


SECOND = """
import os, sys, time
for p in ("maxwellfdm.jl_amd", "oracle", "tests"):
    sys.path.insert(0, os.path.join(sys.argv[1], p))
import numpy as np
import maxwellfdfd as pkg, oracle as O
from conftest import spec_of
from test_gpu_resident import OM, TOL, system
for k in range(3):
    m, rng = system(pkg, (13, 9, 11), (False,) * 3, (0, 0, 0), "diag", 51)
    op = pkg.MaxwellOperator(m, OM)
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
    b = rng.normal(size=A.shape[0]) + 0j
    for _ in range(2):
        t = time.perf_counter()
        e, st = op.solve(b, tol=TOL)
        print("second process: %.2f ms" % (1e3 * (time.perf_counter() - t)), flush=True)
        assert np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
    op.close()
print("second ok", flush=True)
"""


def test_second_process(tmp_path, pkg):
    """A device has one cooperative queue, which the first process that launches so
    holds to its end (this one, here): the solves of a second go on step by step."""
    m, rng = system(pkg, (13, 9, 11), (False,) * 3, (0, 0, 0), "diag", 51)
    op = pkg.MaxwellOperator(m, OM)
    b = rng.normal(size=op.n) + 0j
    op.solve(b, tol=TOL)
    py = tmp_path / "second.py"
    py.write_text(SECOND)
    p = subprocess.run([sys.executable, "-u", str(py), ROOT], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONDONTWRITEBYTECODE="1"))
    print(p.stdout)
    op.solve(b, tol=TOL)
    op.close()
    assert p.returncode == 0 and "second ok" in p.stdout, p.stdout + p.stderr
