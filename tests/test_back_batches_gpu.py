"""Back-contractions of batches of triples (both kinds of term, all row and column tiles) against the FP64 oracle.

Every gradient element is a sum of at most 6 o^2 v^2 FP64 products (per row of an output), in another order than the
oracle's: the bound on the difference, n 2^-53 times the sum of absolute values, stays under 1e-11 of the largest entry
for these sizes (n <= 2e6, terms of random sign)."""

import numpy as np
import pytest

import oracle
from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu
NAMES = ("ovvv", "ovoo", "ovov", "t1", "t2")


def _check(got, want):
    for k in NAMES:
        scale = max(np.abs(want[k]).max(), 1e-300)
        assert np.abs(got[k] - want[k]).max() < 1e-11 * scale, k


# v8 + o8 columns: one tile up to 128, then two; v = 8, 16, 17, 64, 65: edges of row groups, blocks and slabs; o = 8, 9:
# edge of the second operand's columns; 10, 9: more triples than a batch of 128
@pytest.mark.parametrize("o,v", [(2, 8), (3, 16), (8, 17), (9, 15), (10, 9), (3, 64), (2, 65), (2, 119), (2, 121),
                                 (3, 129)])
def test_gradients(o, v):
    print("case", o, v, flush=True)
    ctx = gpu.Context(0)
    x = make_triples_inputs(o, v, 7 * o + v)
    ctx.set_triples_inputs(x, ("fp64",))
    _check(ctx.triples_backward("fp64"), oracle.t_grad(x))


def test_gradients_of_one_virtual_vanish():
    """v = 1: the weights of r3 (4 + 1 + 1 - 6) cancel, so the exact gradients are zero and only rounding is left, in the
    oracle as well. With inputs up to m: |Y| <= (6 (1 + o) + 3) m^2, each gradient sums at most 6 terms of o^2 triples of
    12 |Y| m / D, twice; every term is rounded less than 32 times by 2^-53."""
    o = 2
    ctx = gpu.Context(0)
    x = make_triples_inputs(o, 1, 7 * o + 1)
    ctx.set_triples_inputs(x, ("fp64",))
    m = max(1.0, *(np.abs(a).max() for a in (x.t1, x.t2, x.ovvv, x.ovoo, x.ovov)))
    d = 3.0 * (x.e[o:].min() - x.e[:o].max())
    assert d > 0
    bound = 2 * 6 * o ** 2 * 12 * (6 * (1 + o) + 3) * m ** 3 / d * 32 * 2.0 ** -53
    g, want = ctx.triples_backward("fp64"), oracle.t_grad(x)
    for k in NAMES:
        assert np.abs(g[k]).max() <= bound and np.abs(want[k]).max() <= bound, (k, bound)


@pytest.mark.parametrize("o,v,n", [(6, 10, 3), (4, 33, 5), (3, 7, 40)])
def test_shards_add_up(o, v, n):
    """The batches of every shard hold each of its triples once (n past the number of triples: empty shards)."""
    ctx = gpu.Context(0)
    x = make_triples_inputs(o, v, 3)
    ctx.set_triples_inputs(x, ("fp64",))
    total = None
    for s in range(n):
        ctx.set_shard(s, n)
        g = ctx.triples_backward("fp64")
        total = g if total is None else {k: total[k] + g[k] for k in NAMES}
    _check(total, oracle.t_grad(x))
