"""FP64 (T) at sizes that end in the middle of a group of four fixed indices (v mod 4 = 2, 3, 2) and of a tile: every F_ijk
against the oracle (1e-12 of the largest, as the other FP64 comparisons), the same bits from every way of launching the work,
and the gradients against the oracle's (1e-11 of each one's largest entry)."""

import ctypes

import numpy as np
import pytest

import oracle
from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,seed", [(5, 70, 15), (4, 67, 16), (6, 130, 17)])
def test_launches_give_the_same_bits(o, v, seed):
    print(f"case launches o={o} v={v}", flush=True)
    inp = make_triples_inputs(o, v, seed)
    Eo, Fo = oracle.t_ijk(inp)
    with gpu.Context(0) as ctx:
        ctx.set_triples_inputs(inp, ("fp64",))
        E, F, _ = ctx.triples_forward("fp64", with_F=True)
        assert np.abs(F - Fo).max() <= 1e-12 * np.abs(Fo).max()
        assert abs(E - Eo) <= 1e-12 * abs(Eo)
        for n in (1, 3):  # one or three triples per launch, each with its own queues
            ctx.set_batch(n)
            e, f, _ = ctx.triples_forward("fp64", with_F=True)
            assert e == E and np.array_equal(f, F), n
        e = ctypes.c_double()
        ctx.check(ctx.lib.scess_t_forward_noalloc(ctx.h, gpu.PRECISIONS["fp64"], ctypes.byref(e)))
        assert e.value == E


@pytest.mark.parametrize("o,v,seed", [(3, 70, 8), (4, 40, 9)])
def test_gradients(o, v, seed):
    print(f"case gradients o={o} v={v}", flush=True)
    inp = make_triples_inputs(o, v, seed)
    with gpu.Context(0) as ctx:
        ctx.set_triples_inputs(inp, ("fp64",))
        g = ctx.triples_backward("fp64")
    for k, want in oracle.t_grad(inp).items():
        assert np.abs(g[k] - want).max() <= 1e-11 * np.abs(want).max(), k
