"""Host arrays in and out: copies through the context's slots against device
arrays of the caller, at sizes around the smallest threaded copy (16 MiB, four
threads), with remainders of a slot (1 MiB) and of the threads' rounds, up to
all eight threads (32 MiB), and from several threads at once."""
import threading

import numpy as np
import pytest
import torch

from test_gpu_resident import OM, say, system

pytestmark = pytest.mark.gpu


def pair(pkg, N, seed):
    m, rng = system(pkg, N, (False,) * 3, (0, 0, 0), "diag", seed)
    n = 3 * int(np.prod(N))
    return pkg.MaxwellOperator(m, OM), rng.normal(size=n) + 1j * rng.normal(size=n)


def on_device(op, x):
    xd = torch.from_numpy(x).to("cuda")
    yd = torch.empty_like(xd)
    torch.cuda.synchronize()
    op.apply_dev(xd.data_ptr(), yd.data_ptr(), 1, "fp64")
    return yd.cpu().numpy()


# 48·M bytes: one cell, 16 MiB − 1,216, 16 MiB + 32, 18 MiB, 24 MiB, just below 32 MiB, 35.6 MiB
@pytest.mark.parametrize("N", [(1, 1, 1), (3, 25, 4660), (2, 174763, 1), (64, 64, 96), (64, 64, 128), (19, 67, 549),
                               (95, 91, 90)])
def test_copies(N, pkg):
    """Bitwise: a copy moves bytes."""
    op, x = pair(pkg, N, 1)
    say("copies", N)
    want = on_device(op, x)
    for _ in range(3):   # the second pass reuses blocks and slots
        assert np.array_equal(op.apply(x), want)
    op.close()


def test_copies_threads(pkg):
    """Three threads on one context: one copy at a time has the slots, the
    others copy without them; blocks in use are not handed out twice."""
    work = [pair(pkg, N, 2) for N in ((80, 80, 57), (73, 91, 55), (90, 80, 64))]
    want = [on_device(op, x) for op, x in work]
    bad = []

    def run(k):
        for _ in range(6):
            if not np.array_equal(work[k][0].apply(work[k][1]), want[k]):
                bad.append(k)

    th = [threading.Thread(target=run, args=(k,)) for k in range(3)]
    say("copies from threads")
    for t in th:
        t.start()
    for t in th:
        t.join()
    for op, _ in work:
        op.close()
    assert not bad
