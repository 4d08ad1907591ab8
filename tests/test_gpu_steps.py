"""The step-by-step SQMR solver with its d, z updates put off, against chunks
of one step, which apply every update at once."""
import numpy as np
import pytest

from conftest import spec_of
from test_gpu_resident import OM, TOL, say, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("check_every", [2, 3, 4, 5, 8, 9, 14])
def test_deferred_updates(check_every, precision, pkg, O):
    """Chunks that end at, before and after the put-off steps, a budget inside a
    chunk, right-hand sides that finish at the start (b = 0) and early (a near
    solution as the guess).  After 23 steps from the same state the iterates
    differ by rounding only, which grows less than a thousandfold in that many
    steps of this recurrence: 1e-11 from FP64, 2e-3 from FP32 vectors."""
    m, rng = system(pkg, (21, 13, 11), (False,) * 3, (0, 0, 0), "diag", 12)
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
    n = A.shape[0]
    b = rng.normal(size=(3, n)) + 1j * rng.normal(size=(3, n))
    b[1] = 0
    op = pkg.MaxwellOperator(m, OM)
    op.set_tile("fp64", 4, 4, 1)
    op.set_tile("mixed", 4, 4, 1)
    say("steps", check_every, precision)
    e, _ = op.solve(b, tol=1e-30, maxit=23, check_every=check_every, precision=precision, raise_on_noconv=False)
    e1, _ = op.solve(b, tol=1e-30, maxit=23, check_every=1, precision=precision, raise_on_noconv=False)
    assert np.linalg.norm(e - e1) <= (1e-11 if precision == "fp64" else 2e-3) * np.linalg.norm(e1)
    near, _ = op.solve(b[2], tol=1e-6)
    g = np.zeros_like(b)
    g[2] = near
    e, st = op.solve(b, x0=g, tol=TOL, check_every=check_every, precision=precision)
    op.close()
    assert st.converged and not e[1].any()
    for r in (0, 2):
        assert np.linalg.norm(b[r] - A @ e[r]) <= 1.01 * TOL * np.linalg.norm(b[r])


@pytest.mark.parametrize("N", [(70, 37, 45), (64, 130, 31), (33, 9, 90), (150, 21, 1)])
@pytest.mark.parametrize("scene", ["diag", "mu", "full"])
def test_launch_tiles(N, scene, pkg):
    """Tiles chosen at the launch (short last chunks, several right-hand sides)
    against a fixed shape: each value is formed from the same terms in the same
    order whatever the tile, so they agree to the last bits."""
    m, rng = system(pkg, N, (False, False, N[2] == 1), (0, 0, 0), scene, 4)
    x = rng.normal(size=(3, 3 * int(np.prod(N)))) + 1j * rng.normal(size=(3, 3 * int(np.prod(N))))
    op = pkg.MaxwellOperator(m, OM)
    say("tiles", N, scene)
    y = [op.apply(x), op.apply(x[0])]
    op.set_tile("fp64", 4, 16, 1)
    z = op.apply(x)
    op.close()
    assert np.abs(y[0] - z).max() <= 1e-15 * np.abs(z).max() and np.abs(y[1] - z[0]).max() <= 1e-15 * np.abs(z).max()


@pytest.mark.parametrize("scene", ["diag", "mu", "full"])
@pytest.mark.parametrize("N", [(13, 9, 11), (66, 5, 7), (36, 21, 1)])
def test_bicgstab_products(N, scene, pkg, O):
    """BiCGSTAB, whose inner products end the stencils: every form of the
    stencil (Bloch phases, reflected axes, both tile widths, the direct kernel,
    the sparse product), a right-hand side that starts finished (b = 0)."""
    for bloch, boundft in (((True, True, N[2] == 1), (0, 0, 0)), ((False, False, N[2] == 1), (1, 0, 0)), ((True, False, True), (0, 0, 0))):
        if scene == "full" and any(boundft):
            continue
        m, rng = system(pkg, N, bloch, boundft, scene, 6)
        pkg.set_kbloch(m, [0.02 * v for v in bloch])
        A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
        b = rng.normal(size=(3, A.shape[0])) + 1j * rng.normal(size=(3, A.shape[0]))
        b[1] = 0
        ops = [pkg.MaxwellOperator(m, OM)]
        if scene == "diag":
            ops.append(pkg.MaxwellOperator.from_csc(A))
        if not any(boundft):
            ops.append(pkg.MaxwellOperator(m, OM))
            ops[-1].set_tile("fp64", 0, 1, 0)
        for op in ops:
            say("bicgstab", N, scene, bloch, boundft)
            e, st = op.solve(b, tol=TOL, method="bicgstab")
            op.close()
            assert st.converged and not e[1].any()
            for r in (0, 2):
                assert np.linalg.norm(b[r] - A @ e[r]) <= 1.01 * TOL * np.linalg.norm(b[r])
