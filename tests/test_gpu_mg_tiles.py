"""The one-pass multigrid kernels at the edges of their tiles, bit for bit.

tests/golden/multigrid_tiles_digests.json holds digests of the fields after three steps in
both multigrid modes, made on an MI355X (ROCm 7.2) by this library when every half sweep was
a launch of its own (make_multigrid_digests.run_case on the cases below).  The one-pass
kernels keep every cell update's terms and order, so they have to give the same bits: rows
and planes that do not fill the last tile, one to four z-pairs a thread, walled and periodic
z, coarsening in all three directions, in z alone and in x and y alone, z rows cut into
parts, odd nz below an even level.
"""
import json
import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))

pytestmark = pytest.mark.gpu

# (nx, ny, nz, periodic z, lz)
CASES = [(60, 44, 24, 1, 3.0), (80, 48, 8, 1, 0.7), (40, 24, 10, 0, 2.5), (32, 16, 128, 1, 20.0),
         (64, 32, 8, 0, 40.0), (16, 8, 412, 0, 267.8), (160, 88, 4, 1, 0.5),
         (48, 40, 36, 1, 9.0), (16, 16, 64, 0, 5.0), (96, 48, 6, 0, 1.25)]


@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])))
def test_one_pass_kernels_keep_the_bits(case, precision):
    import make_multigrid_digests as m
    with open(os.path.join(HERE, "golden", "multigrid_tiles_digests.json")) as f:
        want = json.load(f)
    assert (want["steps"], want["seed"]) == (m.STEPS, m.SEED)
    assert m.run_case(*case, precision) == want["digests"][m.key(*case, precision)]
