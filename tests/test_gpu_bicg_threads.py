"""FP64 BiCGSTAB solves of several contexts at the same time, each in a thread of its own: the
bits of a solve alone, with resident kernels that fit side by side and ones that need the whole
device, and small solves that overlap."""
import threading
import time

import numpy as np
import pytest

from gpu_helpers import make_gpu

pytestmark = pytest.mark.gpu


def together(solvers, work):
    """work(solver, index) of every solver in its own thread, started at once; seconds."""
    gate = threading.Barrier(len(solvers) + 1)
    failed = []

    def go(s, q):
        gate.wait()
        try:
            work(s, q)
        except Exception as e:
            failed.append(e)

    threads = [threading.Thread(target=go, args=(s, q)) for q, s in enumerate(solvers)]
    for t in threads:
        t.start()
    gate.wait()
    start = time.perf_counter()
    for t in threads:
        t.join()
    if failed:
        raise failed[0]
    return time.perf_counter() - start


def test_solves_side_by_side_keep_the_bits():
    # resident kernels of 8 to 128 workgroups, two of 256, and launched phases beside them
    sizes = [(128, 64, 4), (64, 64, 4), (150, 41, 25), (128, 128, 32), (256, 128, 32),
             (128, 64, 4), (256, 128, 32), (130, 128, 65)]

    def fresh():
        return [make_gpu(*n, bc="cylinder", maxit=40, tol=1e-30, skip_first=0, seed=q)
                for q, n in enumerate(sizes)]

    alone = fresh()
    for s in alone:
        s.step(3)
    beside = fresh()
    together(beside, lambda s, q: s.step(3))
    for a, b, n in zip(alone, beside, sizes):
        assert np.array_equal(a.xresult(), b.xresult()), n
        for u, v in zip(a.download_velocity(0), b.download_velocity(0)):
            assert np.array_equal(u, v), n
        a.close()
        b.close()


def test_small_solves_overlap():
    # 8 workgroups a context: one after the other, four take four times as long as one; side by
    # side half of that where they share two hardware queues
    solvers = [make_gpu(64, 40, 8, bc="cylinder", maxit=600, tol=1e-30, skip_first=0)
               for _ in range(4)]
    for s in solvers:
        s.step(1)
    one = min(together(solvers[:1], lambda s, q: s.step(1)) for _ in range(5))
    four = min(together(solvers, lambda s, q: s.step(1)) for _ in range(5))
    for s in solvers:
        s.close()
    assert four < 3.0 * one, (four, one)
