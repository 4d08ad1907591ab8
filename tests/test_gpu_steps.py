"""The step-by-step SQMR solver with its d, z updates put off, against chunks
of one step, which apply every update at once."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("window", [(0, 2), (2, 1)])
@pytest.mark.parametrize("N", [(1, 1), (1, 9), (64, 8), (63, 7), (65, 9), (5, 40), (130, 17)])
def test_plane_stencil(N, window, pkg, O):
    """The 2D stencil over the edges of its 64 × 4 tiles: the product and the
    residual norm of a solve against the oracle's A restricted to the window,
    every combination of ends, with and without ε_xy, FP64 and FP32 vectors."""
    N = N + (1,)
    c0, nc = window
    M = int(np.prod(N))
    for bloch in ((False, False, True), (True, False, True), (False, True, True), (True, True, True)):
        for scene in ("diag", "full"):
            m, rng = system(pkg, N, bloch, (0, 0, 0), scene, 7)
            m.εarr[..., 0, 2] = m.εarr[..., 2, 0] = m.εarr[..., 1, 2] = m.εarr[..., 2, 1] = 0
            m.order_cmpfirst = False
            pkg.set_kbloch(m, [0.02 * bloch[0], 0.03 * bloch[1], 0])
            A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)).tocsr()
            A = A[c0 * M:(c0 + nc) * M][:, c0 * M:(c0 + nc) * M]
            x = rng.normal(size=(2, nc * M)) + 1j * rng.normal(size=(2, nc * M))
            op = pkg.MaxwellOperator(m, OM)
            op.set_components(c0, nc)
            say("plane", N, window, bloch, scene)
            want = np.stack([A @ v for v in x])
            # a few sums of about ten products each: 1e-13 of the largest, FP32 storage 1e-6
            assert np.abs(op.apply(x) - want).max() <= 1e-13 * np.abs(want).max()
            xd = torch.from_numpy(x.astype(np.complex64)).to("cuda")
            yd = torch.empty_like(xd)
            torch.cuda.synchronize()
            op.apply_dev(xd.data_ptr(), yd.data_ptr(), 2, "mixed")
            want = np.stack([A @ v for v in xd.cpu().numpy().astype(complex)])
            assert np.abs(yd.cpu().numpy() - want).max() <= 1e-6 * np.abs(want).max()
            e, st = op.solve(x, tol=TOL, method="bicgstab")
            op.close()
            for r in range(2):
                assert np.linalg.norm(x[r] - A @ e[r]) <= 1.01 * TOL * np.linalg.norm(x[r])


def test_plane_steps(pkg, O):
    """SQMR steps on a plane too large for the resident solver (131,072 cells),
    FP64 and mixed, against the oracle's A."""
    N = (431, 350, 1)
    M = int(np.prod(N))
    m, rng = system(pkg, N, (False, False, True), (0, 0, 0), "full", 8)
    m.εarr[..., 0, 2] = m.εarr[..., 2, 0] = m.εarr[..., 1, 2] = m.εarr[..., 2, 1] = 0
    m.order_cmpfirst = False
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)).tocsr()[:2 * M][:, :2 * M]
    op = pkg.MaxwellOperator(m, OM)
    op.set_components(0, 2)
    b = rng.normal(size=2 * M) + 1j * rng.normal(size=2 * M)
    for precision in ("fp64", "mixed"):
        say("plane steps", precision)
        e, st = op.solve(b, tol=TOL, precision=precision)
        assert st.converged and np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
    op.close()
