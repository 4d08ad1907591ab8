"""Numbers of right-hand sides outside 1 … 65,535 are refused before a size is
formed from them, by the C entry points that take host arrays (one cell, where
the wrapped size of −1 right-hand sides would round up to nothing)."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_resident import OM, say, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [(1, 1, 1), (5, 4, 3)])
def test_refused(N, pkg):
    from maxwellfdfd import _lib as L
    m, rng = system(pkg, N, (False,) * 3, (0, 0, 0), "diag", 81)
    op = pkg.MaxwellOperator(m, OM)
    lib = pkg.lib()
    x = rng.normal(size=op.n) + 0j
    want = op.apply(x)
    y, e = np.full_like(x, 7.0), np.full_like(x, 7.0)
    o, st = L.mfd_solve_opts(), L.mfd_solve_stats()
    lib.mfd_solve_opts_default(C.byref(o))
    ms = C.c_double()
    for nrhs in (-1, 0, -(1 << 40), 65536):
        say("refused", N, nrhs)
        assert lib.mfd_op_apply(op._h, L.ptr(x), L.ptr(y), nrhs) == L.MFD_ERR_ARG
        assert lib.mfd_solve(op._h, L.ptr(x), L.ptr(e), nrhs, C.byref(o), C.byref(st)) == L.MFD_ERR_ARG
        assert lib.mfd_op_bench_apply(op._h, nrhs, L.MFD_FP64, 1, C.byref(ms)) == L.MFD_ERR_ARG
    assert (y == 7.0).all() and (e == 7.0).all()
    assert np.array_equal(op.apply(x), want)
    op.close()
