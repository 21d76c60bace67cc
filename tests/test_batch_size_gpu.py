"""The number of triples per launch chosen for small v: E(T) and every F_ijk are those of any other batch, bit for bit."""

import numpy as np
import pytest

from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu


# one batch for all triples; several; the line where the rule stops (v = 100: 40 or 23 triples, 130: 16 or 8)
@pytest.mark.parametrize("o,v", [(2, 5), (14, 19), (5, 33), (6, 100), (4, 130)])
def test_any_batch_gives_the_same(o, v):
    print("case", o, v, flush=True)
    ctx = gpu.Context(0)
    ctx.set_int8_digits(5)
    modes = ("fp64", "fp32", "bf16x3", "ozaki")
    ctx.set_triples_inputs(make_triples_inputs(o, v, o + v), modes)
    for p in modes:
        E, F, _ = ctx.triples_forward(p, with_F=True)
        for n in (1, 8):
            ctx.set_batch(n)
            e, f, _ = ctx.triples_forward(p, with_F=True)
            assert e == E and np.array_equal(f, F), (p, n)
        ctx.set_batch(0)
