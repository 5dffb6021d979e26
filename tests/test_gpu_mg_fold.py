"""The preconditioned iteration's alpha and omega on both sides of the 1024 partials up to which
each block of their users folds them, bit for bit.

tests/golden/multigrid_fold_digests.json holds digests of the fields after three steps in both
multigrid modes, made on an MI355X (ROCm 7.2) by this library when a kernel of one block folded
every scalar (make_multigrid_digests.run_case on the cases below): 1024 and 1088 partials.
"""
import json
import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))

pytestmark = pytest.mark.gpu

CASES = [(256, 128, 32, 1, 0.5), (256, 136, 32, 0, 0.5)]  # (nx, ny, nz, periodic z, lz)


@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])))
def test_folds_keep_the_bits(case, precision):
    import make_multigrid_digests as m
    with open(os.path.join(HERE, "golden", "multigrid_fold_digests.json")) as f:
        want = json.load(f)
    assert (want["steps"], want["seed"]) == (m.STEPS, m.SEED)
    assert m.run_case(*case, precision) == want["digests"][m.key(*case, precision)]
