"""Every box shape and form of the resident solver, on sizes with remainders on
each axis: the trace names the boxes, so a system that falls back to the
step-by-step solver fails here."""
import re

import numpy as np
import pytest

from conftest import spec_of
from test_gpu_resident import OM, TOL, compare, say, system

pytestmark = pytest.mark.gpu


def run(pkg, A, op, b, precision, box, capfd, monkeypatch):
    """Solves, checks the residual on A and that each precision's cycles ran in
    the boxes named (FP32, FP64); the statistics."""
    monkeypatch.setenv("MFD_SOLVE_TRACE", "1")
    capfd.readouterr()
    e, st = op.solve(b, tol=TOL, precision=precision)
    trace = capfd.readouterr().err
    monkeypatch.delenv("MFD_SOLVE_TRACE")
    ran = {m.group(1): m.group(2) for m in re.finditer(r"\[mfd resident\] (fp\d\d) boxes (\S+),", trace)}
    say("ran", ran, st.iterations, st.iterations_fp32)
    assert ran.get("fp32" if precision == "mixed" else "fp64") == box[precision]
    assert st.converged and np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
    return st


# (grid, box of FP64 vectors, box of FP32 vectors with diagonal ε and μ = 1, else)
SOLIDS = [((9, 13, 10), "8x4x4", "8x4x4", "8x4x4"), ((33, 37, 35), "8x8x4", "8x8x4", "8x8x4"),
          ((41, 36, 45), "16x8x4", "16x8x4", "16x8x4"), ((47, 47, 49), "16x8x4", "16x8x4", "16x8x4"),
          ((50, 59, 61), None, "16x8x8", None)]


@pytest.mark.parametrize("N,box64,box32,box32t,scene", [s + (scene,) for s in SOLIDS for scene in ("diag", "mu", "full")
                                                        if scene == "diag" or s[3]])
def test_solids(N, box64, box32, box32t, scene, pkg, O, capfd, monkeypatch):
    box = {"fp64": box64, "mixed": box32 if scene == "diag" else box32t}
    for bloch, boundft in (((False, True, False), (0, 0, 0)), ((True, False, True), (0, 1, 1))):
        if scene == "full" and any(boundft):
            boundft = (0, 0, 0)
        m, rng = system(pkg, N, bloch, boundft, scene, 41)
        A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
        b = rng.normal(size=A.shape[0]) + 1j * rng.normal(size=A.shape[0])
        for precision in ("fp64", "mixed"):
            if box[precision] is None:
                continue
            say("solid", N, scene, bloch, boundft, precision)
            op = pkg.MaxwellOperator(m, OM)
            st = run(pkg, A, op, b, precision, box, capfd, monkeypatch)
            if precision == "fp64":
                op.set_tile("fp64", 4, 4, 1)
                _, step = op.solve(b, tol=TOL)
                compare((st.iterations, step.iterations), (st.outer_cycles, step.outer_cycles))
            op.close()


# planes of cells, the boxes as above
PLANES = [((37, 30), "16x8x1", "16x8x1", "16x8x1"), ((200, 301), "32x16x1", "32x16x1", "32x16x1"),
          ((431, 350), None, "32x32x1", None)]
# a window of the 2D models (its first component, how many), or all three, with what each can have
FORMS = [((0, 2), "diag"), ((0, 2), "full"), ((2, 1), "diag"), ((0, 3), "diag"), ((0, 3), "mu"), ((0, 3), "full")]


@pytest.mark.parametrize("N,box64,box32,box32t,window,scene", [p + f for p in PLANES for f in FORMS if f[1] == "diag" or p[3]])
def test_planes(N, box64, box32, box32t, window, scene, pkg, O, capfd, monkeypatch):
    c0, nc = window
    if nc == 1 and N == (200, 301):
        box64 = None   # the exchange of one component's boxes finds no room
    box = {"fp64": box64, "mixed": box32 if scene == "diag" else box32t}
    M = int(np.prod(N))
    # one-cell z axis: periodic (the 2D models), or closed with all three components
    for bloch in ((False, False, True), (True, False, True)) + (((False, True, False),) if nc == 3 else ()):
        m, rng = system(pkg, N + (1,), bloch, (0, 0, 0), scene, 43)
        m.order_cmpfirst = False
        if nc < 3:
            m.εarr[..., 0, 2] = m.εarr[..., 2, 0] = m.εarr[..., 1, 2] = m.εarr[..., 2, 1] = 0
        A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)).tocsr()[c0 * M:(c0 + nc) * M][:, c0 * M:(c0 + nc) * M]
        b = rng.normal(size=nc * M) + 1j * rng.normal(size=nc * M)
        for precision in ("fp64", "mixed"):
            if box[precision] is None:
                continue
            say("plane", N, scene, window, bloch, precision)
            op = pkg.MaxwellOperator(m, OM)
            if nc < 3:
                op.set_components(c0, nc)
            st = run(pkg, A, op, b, precision, box, capfd, monkeypatch)
            if precision == "fp64":
                op.set_tile("fp64", 4, 4, 1)
                _, step = op.solve(b, tol=TOL)
                compare((st.iterations, step.iterations), (st.outer_cycles, step.outer_cycles))
            op.close()
