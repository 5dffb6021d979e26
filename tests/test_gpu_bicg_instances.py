"""Every instance of the resident BiCGSTAB kernel, bit for bit against the oracle: both operators,
tiles of at most 256 and 512 cells and halves of larger ones, uniform whole blocks and others;
halves of several tiles, which exchange rows, up to the largest grid of whole tiles; and last
blocks of one to seven planes marching down and up, whole and in halves."""
import numpy as np
import pytest

from gpu_helpers import fields_equal, make_pair

pytestmark = pytest.mark.gpu

# nx = 8 * even + r ends with r planes marching down, 8 * odd + r marching up
ENDS = [16 + r for r in range(1, 8)] + [24 + r for r in range(1, 8)]
# (nx, ny, nz), boundary conditions, precond, iterations
CASES = (
    # uniform: 256 and 512 cells, halves of one, two and four tiles
    [((n, 64, 4), "cylinder", p, 10) for n in (16, 24) for p in (0, 1)]
    + [((n, 64, 8), "slip", p, 10) for n in (16, 24) for p in (0, 1)]
    + [((16, 64, 16), "slip", 1, 10), ((32, 64, 32), "cylinder", 0, 10),
       ((32, 64, 32), "cylinder", 1, 10), ((24, 128, 32), "slip", 0, 10),
       ((256, 128, 32), "cylinder", 0, 5), ((256, 128, 32), "cylinder", 1, 5)]
    # others, by their last block
    + [((n, 43, 5), "slip", n % 2, 8) for n in ENDS]
    + [((n, 37, 12), "cylinder", n // 2 % 2, 8) for n in ENDS]
    + [((n, 41, 25), "cylinder", n % 2, 8) for n in ENDS]
    + [((n, 41, 25), "slip", 1 - n % 2, 8) for n in ENDS]
)


@pytest.mark.parametrize("n,bc,precond,maxit", CASES,
                         ids=["x".join(map(str, c[0])) + f"-{c[1]}-{c[2]}" for c in CASES])
def test_instance_bitwise(n, bc, precond, maxit):
    gpu, sim, o, g = make_pair(*n, bc=bc, precond=precond, maxit=maxit, tol=1e-30, skip_first=0)
    for s in range(2):
        a, b = gpu.step(1), sim.step()
        for key in ("iters", "err", "cd", "cl", "cfl"):
            assert a[key] == b[key] or (np.isnan(a[key]) and np.isnan(b[key])), (s, key, a, b)
        assert fields_equal(gpu, sim) == [], s
    assert gpu.resident_solve() == 0
    gpu.close()
