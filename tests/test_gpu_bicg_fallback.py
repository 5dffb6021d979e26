"""A resident BiCGSTAB solve that gives up, bit for bit against the oracle: in its first launch,
and in its second after 1024 iterations have advanced x and the solver's state; then further
solves, which take launched phases from the start.  Every block gives up after its first wait,
so the kernel ends normally."""
import numpy as np
import pytest

from gpu_helpers import fields_equal, make_pair

pytestmark = pytest.mark.gpu


# (nx, ny, nz): whole march blocks, halves of them; most iterations, launches before the one
# that gives up
@pytest.mark.parametrize("n,maxit,launches", [
    ((40, 16, 4), 12, 0), ((19, 41, 25), 12, 0), ((40, 16, 4), 1100, 1), ((33, 35, 16), 1030, 1),
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
@pytest.mark.parametrize("precond", [0, 1])
def test_solve_begins_again_by_launched_phases(n, maxit, launches, precond):
    gpu, sim, o, g = make_pair(*n, bc="cylinder", precond=precond, maxit=maxit, tol=1e-30,
                               skip_first=0)
    assert gpu.resident_solve() == 0
    for s in range(3):
        if s == 1:
            gpu.resident_solve(launches)
        a, b = gpu.step(1), sim.step()
        for key in ("iters", "err", "cd", "cl", "cfl"):
            assert a[key] == b[key] or (np.isnan(a[key]) and np.isnan(b[key])), (s, key, a, b)
        assert fields_equal(gpu, sim) == [], s
        assert gpu.resident_solve(launches if s else -1) == (1 if s else 0)
    gpu.close()


def test_a_grid_the_kernel_does_not_take_never_falls_back():
    gpu, sim, o, g = make_pair(16, 10, 129, bc="slip", maxit=3, tol=1e-30, skip_first=0)
    gpu.resident_solve(0)
    gpu.step(1)
    sim.step()
    assert fields_equal(gpu, sim) == []
    assert gpu.resident_solve() == 0
    gpu.close()
