"""The red-black pass of two sweeps where it can go wrong, bit for bit against the oracle: rows
whole (walled, periodic) and cut into pieces of pairs, one tile of rows and several, short and
partly filled last spans of planes and tiles, solves that end after an odd and an even sweep, by
their count and by their tolerance, and odd rows, which take the half sweeps."""
import numpy as np
import pytest

from gpu_helpers import fields_equal, make_pair

pytestmark = pytest.mark.gpu

# (nx, ny, nz), boundary conditions, most sweeps, tolerance
CASES = [
    ((8, 8, 4), "cylinder", 7, 1e-30), ((4, 4, 4), "slip", 1, 1e-30),
    ((5, 9, 4), "slip", 2, 1e-30), ((13, 90, 6), "cylinder", 9, 1e-30),
    ((21, 33, 8), "slip", 10, 1e-30), ((10, 300, 34), "cylinder", 5, 1e-30),
    ((9, 130, 60), "slip", 6, 1e-30), ((7, 150, 64), "cylinder", 5, 1e-30),
    ((12, 40, 120), "cylinder", 6, 1e-30), ((6, 31, 202), "slip", 5, 1e-30),
    ((40, 20, 10), "slip", 70, 1e-30), ((24, 16, 6), "cylinder", 400, 2e-4),
    ((24, 16, 6), "slip", 400, 3e-4), ((24, 18, 6), "cylinder", 400, 1e-4),
    ((24, 16, 5), "slip", 5, 1e-30),
]


@pytest.mark.parametrize("n,bc,maxit,tol", CASES,
                         ids=["x".join(map(str, c[0])) + f"-{c[1]}-{c[2]}-{c[3]}" for c in CASES])
def test_sor_pass_bitwise(n, bc, maxit, tol):
    gpu, sim, o, g = make_pair(*n, bc=bc, solver=1, maxit=maxit, tol=tol, skip_first=0)
    for s in range(3):
        a, b = gpu.step(1), sim.step()
        for key in ("iters", "err", "cd", "cl", "cfl"):
            assert a[key] == b[key] or (np.isnan(a[key]) and np.isnan(b[key])), (s, key, a, b)
        assert fields_equal(gpu, sim) == [], s
    gpu.close()
