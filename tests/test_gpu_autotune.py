"""The tile autotuner: operators whose stencil has no tiles keep the rule's shape,
the others a shape of the candidates, and the product stays the same."""
import numpy as np
import pytest

from conftest import spec_of
from test_gpu_resident import OM, say, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window", [(0, 2), (2, 1)])
def test_window(window, pkg, O):
    """One plane has one plane per tile by the rule; the sweep's 4 to 32 would be
    noise between runs of one kernel."""
    N = (70, 61)
    c0, nc = window
    M = int(np.prod(N))
    m, rng = system(pkg, N + (1,), (False, False, True), (0, 0, 0), "diag", 61)
    m.order_cmpfirst = False
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)).tocsr()[c0 * M:(c0 + nc) * M][:, c0 * M:(c0 + nc) * M]
    x = rng.normal(size=nc * M) + 1j * rng.normal(size=nc * M)
    op = pkg.MaxwellOperator(m, OM)
    op.set_components(c0, nc)
    y = op.apply(x)
    for _ in range(2):
        say("window", window)
        t64, t32, ms = op.autotune(1, 2)
        assert tuple(t64) == tuple(t32) and t64[1] == 1 and min(ms) > 0
        assert np.array_equal(op.apply(x), y)
    op.set_tile("fp64", 4, 4, 1)   # the marching stencil, until it is tuned again
    op.autotune(1, 2)
    assert np.array_equal(op.apply(x), y)
    op.close()
    # a few sums of about ten products each
    assert np.abs(y - A @ x).max() <= 1e-13 * np.abs(y).max()


def test_solid(pkg, O):
    m, rng = system(pkg, (37, 21, 19), (False,) * 3, (0, 0, 0), "diag", 62)
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
    x = rng.normal(size=A.shape[0]) + 1j * rng.normal(size=A.shape[0])
    op = pkg.MaxwellOperator(m, OM)
    op.set_tile("fp64", 0, 1, 0)   # the direct kernel is no candidate
    t64, t32, ms = op.autotune(1, 2)
    say("solid", t64, t32, ms)
    assert t64[0] in (1, 2, 4, 8) and t32[0] in (1, 2, 4, 8) and min(ms) > 0
    y = op.apply(x)
    op.close()
    assert np.abs(y - A @ x).max() <= 1e-13 * np.abs(y).max()
