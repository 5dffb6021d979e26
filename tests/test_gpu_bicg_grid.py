"""The resident BiCGSTAB kernel where it can go wrong, bit for bit against the oracle: tiles of
at most 256 and 512 cells and just above, whole and partly filled, last blocks of one to seven
planes in either marching direction (whole blocks and halves), walled and periodic z, both
operators, a solve of more than one launch, and the sizes on either side of the most blocks
it takes (above them the launched phases run)."""
import numpy as np
import pytest

from gpu_helpers import fields_equal, make_pair

pytestmark = pytest.mark.gpu

# (nx, ny, nz), boundary conditions, precond, iterations
CASES = [
    ((16, 64, 4), "cylinder", 0, 12), ((64, 64, 4), "slip", 1, 12), ((17, 43, 6), "slip", 0, 12),
    ((24, 64, 8), "cylinder", 1, 12), ((31, 17, 30), "slip", 0, 12),
    ((33, 57, 9), "cylinder", 0, 12), ((16, 64, 16), "cylinder", 0, 12),
    ((9, 33, 31), "slip", 0, 12), ((10, 41, 32), "cylinder", 1, 12),
    ((19, 41, 25), "slip", 0, 12), ((20, 33, 32), "cylinder", 0, 12),
    ((13, 30, 70), "cylinder", 0, 12), ((30, 40, 64), "slip", 1, 12),
    ((16, 9, 128), "cylinder", 0, 12), ((16, 10, 129), "slip", 0, 12),
    ((1024, 19, 27), "cylinder", 0, 4), ((1025, 19, 27), "slip", 0, 4),
    ((40, 16, 4), "cylinder", 0, 1100),
]


@pytest.mark.parametrize("n,bc,precond,maxit", CASES,
                         ids=["x".join(map(str, c[0])) + f"-{c[2]}" for c in CASES])
def test_resident_solve_bitwise(n, bc, precond, maxit):
    gpu, sim, o, g = make_pair(*n, bc=bc, precond=precond, maxit=maxit, tol=1e-30, skip_first=0)
    for s in range(2):
        a, b = gpu.step(1), sim.step()
        for key in ("iters", "err", "cd", "cl", "cfl"):
            assert a[key] == b[key] or (np.isnan(a[key]) and np.isnan(b[key])), (s, key, a, b)
        assert fields_equal(gpu, sim) == [], s
    gpu.close()
