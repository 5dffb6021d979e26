"""The one-pass multigrid kernels with two and four z-pairs a thread, bit for bit: walled and
periodic z, whole rows and rows cut into parts, coarsening in z alone and in all directions; in
double, walled levels with one.

tests/golden/multigrid_pairs_digests.json holds digests of the fields after three steps in both
multigrid modes, made on an MI355X (ROCm 7.2) by this library when every half sweep was a launch
of its own (make_multigrid_digests.run_case on the cases below).
"""
import json
import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))

pytestmark = pytest.mark.gpu

# (nx, ny, nz, periodic z, lz): the first level of each has two pairs (128x64) or, in float, four
# (128x96) a thread; rows of 48 pairs are whole, longer ones cut; the longer lz is of cells as
# wide as high, the shorter of flat ones, which coarsen in z alone
CASES = [(nx, ny, nz, zper, lz) for nx, ny, nz, lzs in (
    (128, 64, 96, (15.0, 1.5)), (128, 64, 192, (30.0, 3.0)), (128, 96, 96, (15.0, 1.5)),
    (128, 96, 256, (40.0, 4.0))) for lz in lzs for zper in (0, 1)]


@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_pairs_keep_the_bits(case, precision):
    import make_multigrid_digests as m
    with open(os.path.join(HERE, "golden", "multigrid_pairs_digests.json")) as f:
        want = json.load(f)
    assert (want["steps"], want["seed"]) == (m.STEPS, m.SEED)
    assert m.run_case(*case, precision) == want["digests"][m.key(*case, precision)]
