"""flops_executed of the FP64 (T) forward: the 16 x 16 x 4 MFMAs of the W-build, counted one by one here."""

import pytest

from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v", [(2, 5), (5, 16), (4, 33), (17, 20), (3, 98)])
def test_fp64_counts_the_issued_mfmas(o, v):
    blocks = len(range(0, v, 16)) ** 2
    fixed = 4 * len(range(0, v, 4))                                # fixed indices in groups of four
    steps_f, steps_m = len(range(0, v, 4)), len(range(0, o, 4))   # k-steps of an f-term and of an m-term
    mfma = 0
    for i in range(o):
        for j in range(i + 1):
            for k in range(j + 1):
                if i == j == k:
                    continue
                terms = 6 if i != j and j != k else 3  # of either kind; two equal indices: half of them
                mfma += terms * (steps_f + steps_m) * blocks * fixed
    with gpu.Context(0) as ctx:
        ctx.set_triples_inputs(make_triples_inputs(o, v, 1), ("fp64",))
        _, stats = ctx.triples_forward("fp64")
    assert stats["flops_executed"] == mfma * 2 * 16 * 16 * 4
