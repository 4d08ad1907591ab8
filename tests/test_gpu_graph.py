"""The chunk graph a workspace keeps from call to call, where the scratch of
the two-pass direct kernel (in the graph's launches) has been replaced since:
an apply of more right-hand sides than before needs a larger one."""
import numpy as np
import pytest
import torch

from conftest import spec_of
from test_gpu_resident import OM, TOL, say, system

pytestmark = pytest.mark.gpu


def direct(pkg, O, N, kind, seed):
    """An operator that the direct kernel serves, and the oracle's A."""
    m, rng = system(pkg, N, (False,) * 3, (0, 0, 0), "full" if kind == "mu+full" else "diag", seed)
    if kind == "mu+full":
        for c in range(3):
            m.μarr[..., c, c] = 1 + rng.random(N)
    op = pkg.MaxwellOperator(m, OM)
    if kind == "tile":
        op.set_tile("fp64", 0, 1, 0)
    return op, O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)), rng


@pytest.mark.parametrize("kind", ["mu+full", "tile"])
@pytest.mark.parametrize("method", ["sqmr", "cocg", "bicgstab", "batch"])
def test_scratch_replaced(method, kind, pkg, O):
    made = [direct(pkg, O, N, kind, 21 + k) for k, N in enumerate([(13, 11, 9), (10, 14, 7)])]
    bs = [rng.normal(size=A.shape[0]) + 1j * rng.normal(size=A.shape[0]) for _, A, rng in made]

    def check():
        if method == "batch":
            es = pkg.solve_batch([op for op, _, _ in made], bs, tol=TOL)[0]
        else:
            es = [op.solve(b, tol=TOL, method=method)[0] for (op, _, _), b in zip(made, bs)]
        for (_, A, _), b, e in zip(made, bs, es):
            assert np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)

    for nrhs in (1, 3, 5):
        say("scratch", method, kind, nrhs)
        for op, A, rng in made:
            x = rng.normal(size=(nrhs, A.shape[0])) + 0j
            y = op.apply(x)
            # a few sums of about ten products each
            assert np.abs(y - np.stack([A @ v for v in x])).max() <= 1e-13 * np.abs(y).max()
        # memory that the replaced scratch may have given back is another's now
        held = [torch.full((3 * 13 * 11 * 9,), 7.0, dtype=torch.complex128, device="cuda") for _ in range(8)]
        torch.cuda.synchronize()
        check()
        check()
        assert all(bool((t == 7.0).all()) for t in held)
    for op, _, _ in made:
        op.close()
