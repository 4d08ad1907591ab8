"""Grids whose x-y plane alone has more 4-row tiles than a reduction has partial
sums: rows grow to 8, and where no tile is large enough the direct kernel
serves (the grad-div form, which has none, is refused)."""
import numpy as np
import pytest

from conftest import spec_of
from test_gpu_resident import OM, TOL, say, system

pytestmark = pytest.mark.gpu


def test_many_rows(pkg, O):
    N = (2, 140001, 1)
    m, rng = system(pkg, N, (False, False, True), (0, 0, 0), "diag", 31)
    A = O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr))
    b = rng.normal(size=A.shape[0]) + 1j * rng.normal(size=A.shape[0])
    op = pkg.MaxwellOperator(m, OM)
    for tile in (None, (4, 1, 3), (1, 1, 1)):   # 32-wide of 8 rows: 17,501 tiles; 64-wide of 8 rows: none fits
        if tile:
            op.set_tile("fp64", *tile)
        say("many rows", tile)
        y = op.apply(b)
        assert np.abs(y - A @ b).max() <= 1e-13 * np.abs(y).max()   # sums of about ten products each
        for method in ("sqmr", "cocg", "bicgstab"):
            say("  ", method)
            e, st = op.solve(b, tol=TOL, method=method)
            assert st.converged and np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
    op.set_graddiv(True)
    with pytest.raises(pkg.MfdError):
        op.solve(b, tol=TOL)
    op.set_graddiv(False)
    e, st = op.solve(b, tol=TOL)
    op.close()
    assert st.converged and np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
