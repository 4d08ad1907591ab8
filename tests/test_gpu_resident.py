"""The resident solver (a chunk of SQMR steps in one kernel) over the edges of
its boxes, for every form it serves: converged solves whose residual is taken
on the oracle's A, and the step counts of the step-by-step solver, which an
operator with a hand-set tile runs."""
import sys
import threading

import numpy as np
import pytest

from conftest import spec_of

pytestmark = pytest.mark.gpu

def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def system(pkg, N, bloch, boundft, scene, seed):
    rng = np.random.default_rng(seed)
    m = pkg.ModelFull(pkg.Grid([np.cumsum(np.r_[0.0, 1 + 0.2 * rng.random(n)]) for n in N], bloch))
    pkg.set_ωpml(m, OM)
    npml = tuple(2 if n >= 8 and not b else 0 for n, b in zip(N, bloch))
    pkg.set_Npml(m, (npml, npml))
    pkg.set_boundft(m, boundft)
    eps = np.zeros(N + (3, 3), complex, order="F")
    mu = np.zeros_like(eps)
    for c in range(3):
        eps[..., c, c] = 2 + 4 * rng.random(N) - 2j
        mu[..., c, c] = 1 + rng.random(N) if scene == "mu" else 1
    if scene == "full":
        for v, w in ((0, 1), (0, 2), (1, 2)):
            eps[..., v, w] = eps[..., w, v] = 0.3 * rng.normal(size=N)
    m.εarr, m.μarr = eps, mu
    return m, rng


# one box and less, its edges on each axis, several boxes with remainders, one
# cell per thread and two (the last two sizes; FP32 also four), one-cell axes
SIZES = [(8, 4, 4), (9, 5, 5), (7, 3, 3), (17, 9, 4), (1, 6, 5), (6, 1, 7), (33, 17, 13), (40, 33, 36), (49, 50, 51)]


TOL = 1e-9
OM = 0.3   # with the lossy ε below, systems that SQMR solves at every size used


def compare(its, cycles):
    """The two solvers run the same recurrences in another order of summation:
    as many refinement cycles, and step counts within what rounding moves
    them.  A wrong operator or halo in the resident kernel would part its
    recurrence from the true residual and cost cycles, or not converge."""
    assert abs(cycles[0] - cycles[1]) <= 1
    assert its[0] <= 1.25 * its[1] + 64 and its[1] <= 1.25 * its[0] + 64


@pytest.mark.parametrize("scene", ["diag", "mu", "full"])
@pytest.mark.parametrize("N", SIZES)
def test_resident_solves(N, scene, pkg, O):
    for bloch, boundft in (((False,) * 3, (0, 0, 0)), ((True, False, True), (0, 0, 0)), ((False,) * 3, (1, 0, 1))):
        if scene == "full" and any(boundft):
            continue
        m, rng = system(pkg, N, bloch, boundft, scene, 3)
        A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
        n = A.shape[0]
        b = rng.normal(size=(2, n)) + 1j * rng.normal(size=(2, n))
        for precision in ("fp64", "mixed"):
            say("resident", N, scene, bloch, boundft, precision)
            its, cycles = [], []
            for tile in (None, (4, 4, 1)):
                op = pkg.MaxwellOperator(m, OM)
                if tile:
                    op.set_tile("fp64", *tile)
                    op.set_tile("mixed", *tile)
                e, st = op.solve(b, tol=TOL, precision=precision)
                op.close()
                for r in range(2):
                    assert np.linalg.norm(b[r] - A @ e[r]) <= 1.01 * TOL * np.linalg.norm(b[r])
                its.append(st.iterations)
                cycles.append(st.outer_cycles)
            say("  steps", its, "cycles", cycles)
            if precision == "fp64":   # FP32 cycles stagnate where their rounding takes them
                compare(its, cycles)


@pytest.mark.parametrize("N", [(16, 8), (33, 17), (90, 61)])
@pytest.mark.parametrize("kind", ["TE", "TM"])
def test_resident_window(N, kind, pkg):
    from maxwellfdfd import twod as T
    rng = np.random.default_rng(4)
    g = T.Grid2([np.arange(n + 1.0) for n in N])
    m = (T.ModelTE if kind == "TE" else T.ModelTM)(g)
    T.set_ωpml(m, OM)
    T.set_Npml(m, ((3, 3), (3, 3)))
    eps = np.zeros(N + (1, 3, 3), complex, order="F")
    mu = np.zeros_like(eps)
    for c in range(3):
        eps[..., c, c] = 2 + 4 * rng.random(N + (1,)) - 2j
        mu[..., c, c] = 1
    if kind == "TE":
        eps[..., 0, 1] = eps[..., 1, 0] = 0.3 * rng.normal(size=N + (1,))
    m.m3.εarr, m.m3.μarr = eps, mu
    A = T.create_A(0, OM, m)
    its, cycles = [], []
    for tile in (None, (4, 4, 1)):
        op = T.MaxwellOperator2D(m, OM)
        assert op.windowed
        if tile:
            op.op.set_tile("fp64", *tile)
        b = np.random.default_rng(5).normal(size=op.n) + 0j
        e, st = op.solve(b, tol=TOL)
        op.close()
        assert np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
        its.append(st.iterations)
        cycles.append(st.outer_cycles)
    say("resident window", N, kind, its, cycles)
    compare(its, cycles)


@pytest.mark.parametrize("check_every", [1, 7, 32])
def test_resident_chunks(check_every, pkg, O):
    """Any chunk length, and a budget that ends inside a chunk."""
    m, rng = system(pkg, (20, 13, 11), (False,) * 3, (0, 0, 0), "diag", 8)
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
    b = rng.normal(size=A.shape[0]) + 1j * rng.normal(size=A.shape[0])
    its, cycles = [], []
    for tile in (None, (4, 4, 1)):
        op = pkg.MaxwellOperator(m, OM)
        if tile:
            op.set_tile("fp64", *tile)
        e, st = op.solve(b, tol=TOL, check_every=check_every)
        assert st.converged and np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
        its.append(st.iterations)
        cycles.append(st.outer_cycles)
        e, st = op.solve(b, tol=1e-30, maxit=45, check_every=check_every, raise_on_noconv=False)
        assert st.iterations == 45
        op.close()
    say("resident converged", check_every, its)
    compare(its, cycles)


def test_resident_two_contexts(pkg):
    """Two threads, each with its own context (stream), solving at once."""
    import ctypes as C
    from maxwellfdfd import _lib as L
    m, rng = system(pkg, (24, 20, 22), (False,) * 3, (0, 0, 0), "diag", 9)
    n = 3 * 24 * 20 * 22
    b = rng.normal(size=n) + 1j * rng.normal(size=n)
    lib = pkg.lib()

    def run(out, k):
        ctx, h = C.c_void_p(), C.c_void_p()
        assert lib.mfd_ctx_create(0, C.byref(ctx)) == 0
        g = m._desc()
        assert lib.mfd_op_create(ctx, C.byref(g), 0, L.cplx(OM), L.ptr(m.εarr), L.ptr(m.μarr), C.byref(h)) == 0
        o = L.mfd_solve_opts()
        lib.mfd_solve_opts_default(C.byref(o))
        o.tol, o.maxit = 1e-30, 320
        st = L.mfd_solve_stats()
        res = []
        for _ in range(4):
            e = np.zeros(n, complex)
            rc = lib.mfd_solve(h, L.ptr(b), L.ptr(e), 1, C.byref(o), C.byref(st))
            res.append((rc, e))
        lib.mfd_op_destroy(h)
        lib.mfd_ctx_destroy(ctx)
        out[k] = res

    alone, both = {}, {}
    run(alone, 0)
    th = [threading.Thread(target=run, args=(both, k)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(2):
        for rc, e in both[k]:
            assert rc == L.MFD_ERR_NOCONV and np.array_equal(e, alone[0][0][1])
