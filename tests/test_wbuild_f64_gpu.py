"""The FP64 W-build at the edges of its tiles, k-steps and work queue, against the oracle: F_ijk of every unique
occupied triple. Tolerance: 1e-12 of the largest |F|, as the other FP64 comparisons (FP64 products and sums of at most
4 (v + o) terms on both sides, in another order)."""

import numpy as np
import pytest

import oracle
from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu


# v: one block, an edge of one row, 1 to 4 blocks per tile, uneven halves, several tiles (64 | 65, 112 | 113, 144);
# v mod 4 = 1, 2, 3 (dead fixed indices, k-steps of the last chunk); o: 1 to 4 k-steps of the m-terms, more than a chunk
@pytest.mark.parametrize("o,v,seed", [(2, 2, 1), (2, 16, 2), (3, 17, 3), (5, 31, 4), (9, 34, 5), (13, 49, 6), (17, 20, 7),
                                      (4, 64, 8), (3, 65, 9), (3, 113, 10), (2, 144, 11)])
def test_f_ijk_at_tile_edges(o, v, seed):
    print(f"case wbuild f64 o={o} v={v}", flush=True)
    inp = make_triples_inputs(o, v, seed)
    Eo, Fo = oracle.t_ijk(inp)
    with gpu.Context(0) as ctx:
        ctx.set_triples_inputs(inp, ("fp64",))
        E, F, _ = ctx.triples_forward("fp64", with_F=True)
        ctx.set_batch(3)  # more launches, fewer items each
        E3, F3, _ = ctx.triples_forward("fp64", with_F=True)
    assert np.abs(F - Fo).max() <= 1e-12 * max(np.abs(Fo).max(), 1e-300)
    assert abs(E - Eo) <= 1e-12 * max(abs(Eo), 1e-300)
    assert E3 == E and np.array_equal(F3, F)
