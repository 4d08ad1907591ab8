"""Batches of problems that run step by step, whose chunk graphs share two streams:
the same steps as the single solves, also beside resident problems and from two
threads of one context."""
import threading

import numpy as np
import pytest

from conftest import spec_of
from test_gpu_resident import OM, TOL, say, system

pytestmark = pytest.mark.gpu


def problems(pkg, O, sizes, seed):
    """Operators, right-hand sides, the oracle's A and the single solves' iterates."""
    ops, bs, As = [], [], []
    for k, N in enumerate(sizes):
        m, rng = system(pkg, N, (False,) * 3, (0, 0, 0), "diag", seed + k)
        ops.append(pkg.MaxwellOperator(m, OM))
        As.append(O.to_scipy(O.create_A(spec_of(m), OM, m.εarr, m.μarr)))
        bs.append(rng.normal(size=ops[-1].n) + 1j * rng.normal(size=ops[-1].n))
    return ops, bs, As


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("sizes", [[(70, 45, 44), (53, 52, 51)], [(70, 45, 44), (12, 11, 13), (53, 52, 51), (66, 48, 43), (9, 9, 9)]])
def test_batch(sizes, precision, pkg, O):
    ops, bs, As = problems(pkg, O, sizes, 91)
    say("batch", sizes, precision)
    alone = [op.solve(b, tol=TOL, precision=precision)[0] for op, b in zip(ops, bs)]
    for _ in range(2):   # the second with the kept graphs
        es, st = pkg.solve_batch(ops, bs, tol=TOL, precision=precision)
        for A, b, e, x in zip(As, bs, es, alone):
            assert np.linalg.norm(b - A @ e) <= 1.01 * TOL * np.linalg.norm(b)
            if precision == "fp64":
                assert np.array_equal(e, x)   # the same launches on the same data
    for op in ops:
        op.close()


def test_two_threads(pkg, O):
    work = [problems(pkg, O, sizes, seed) for sizes, seed in (([(70, 45, 44), (53, 52, 51)], 101), ([(66, 48, 43), (57, 49, 50)], 111))]
    want = [pkg.solve_batch(ops, bs, tol=TOL)[0] for ops, bs, _ in work]
    bad = []

    def run(k):
        for _ in range(3):
            es, _ = pkg.solve_batch(work[k][0], work[k][1], tol=TOL)
            bad.extend(k for e, x in zip(es, want[k]) if not np.array_equal(e, x))

    say("two threads")
    th = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for ops, _, _ in work:
        for op in ops:
            op.close()
    assert not bad
