"""Conv-diff with marches of one, two, four and eight planes (the smallest grids take one), last
marches partly filled, with and without the eddy viscosity, bit for bit against the oracle."""
import numpy as np
import pytest

from gpu_helpers import fields_equal, make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bc,cs", [
    ((13, 9, 4), "slip", 0.0), ((24, 20, 6), "cylinder", 0.1), ((131, 128, 16), "cylinder", 0.0),
    ((129, 130, 16), "slip", 0.1), ((197, 93, 31), "cylinder", 0.0), ((257, 128, 32), "slip", 0.0),
    ((130, 160, 40), "cylinder", 0.18), ((41, 512, 64), "slip", 0.0),
], ids=lambda p: "x".join(map(str, p)) if isinstance(p, tuple) else str(p))
def test_marches_bitwise(n, bc, cs):
    gpu, sim, o, g = make_pair(*n, bc=bc, maxit=2, tol=1e-30, skip_first=0, smag_cs=cs)
    for s in range(2):
        a, b = gpu.step(1), sim.step()
        for key in ("cfl", "cd", "cl"):
            assert a[key] == b[key] or (np.isnan(a[key]) and np.isnan(b[key])), (s, key, a, b)
        assert fields_equal(gpu, sim) == [], s
    gpu.close()
