"""The closed-form assembly of A over the sizes where its slots and blocks can
go wrong, against the oracle's A."""
import numpy as np
import pytest

from conftest import spec_of
from test_gpu_parity import assert_csc_equal, rand_params
from test_gpu_resident import say

pytestmark = pytest.mark.gpu


# axes of one and two cells (wrapped neighbours coincide), cells just below, at
# and above a block (128) and a group of blocks (1024), a long axis
@pytest.mark.parametrize("N", [(1, 1, 1), (1, 2, 3), (2, 2, 2), (2, 1, 5), (127, 1, 1), (16, 4, 2), (43, 3, 1),
                               (32, 32, 1), (25, 41, 1), (11, 3, 31), (700, 2, 2)])
@pytest.mark.parametrize("bloch", [(False,) * 3, (True,) * 3, (True, False, True)])
def test_A_slots(N, bloch, pkg, O):
    """Structure and placement exact, values to 1e-13 of the largest: both
    formulations, both orders of the unknowns, mixed boundaries, with and
    without corner terms and the ω² term (ω = 0 keeps structural zeros)."""
    rng = np.random.default_rng(sum(N))
    for boundft, cmpfirst in (((0, 0, 0), True), ((1, 0, 1), False)):
        m = pkg.ModelFull(pkg.Grid([np.cumsum(np.r_[0.0, 1 + 0.2 * rng.random(n)]) for n in N], bloch))
        m.order_cmpfirst = cmpfirst
        pkg.set_boundft(m, boundft)
        pkg.set_kbloch(m, [0.3 * b for b in bloch])
        for ft, full, om in ((0, True, 0.7), (0, False, 0.7), (0, True, 0.0), (1, False, 0.7)):
            say("A slots", N, bloch, boundft, cmpfirst, ft, full, om)
            eps, mu = rand_params(m, 9, full=full, mu=True)
            if ft == 1:   # the ω² term is μ's: corner terms there
                mu[..., 0, 1] = mu[..., 1, 0] = 0.2 * rng.normal(size=N)
            got = pkg.A_csc(m, om, eps, mu, ft=ft)
            assert_csc_equal(got, O.create_A(spec_of(m), om, eps, mu, ft=ft), 1e-13, "A")
