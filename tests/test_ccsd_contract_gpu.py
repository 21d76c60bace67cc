"""One CCSD update where its contractions run in one launch each, straight from the operands (small systems), and
around the line to the GEMM path, against the oracle: 1e-11 of the largest amplitude (FP64 sums of at most o v^2 terms in
another order, as the other updates)."""

import numpy as np
import pytest

from oracle import ccsd_oracle as co
from scess_amd import gpu
from scess_amd.synthetic import _draw, full_eri_chem

pytestmark = pytest.mark.gpu


# (1, 1) and (1, 7): extents of one, one lane per element; (5, 24): a summed extent past one table of 2048 offsets
# (o v^2 = 2880); (6, 36): products on both sides of the line
@pytest.mark.parametrize("o,v,seed,chol", [(1, 1, 1, False), (1, 7, 2, True), (3, 2, 3, False), (5, 24, 4, False),
                                           (5, 24, 4, True), (6, 36, 5, True)])
def test_small_update_matches_oracle(o, v, seed, chol):
    print(f"case ccsd contract o={o} v={v} chol={chol}", flush=True)
    e, L, _ = _draw(o, v, seed)
    L = L * 0.3
    eri = full_eri_chem(L)
    O, V = slice(0, o), slice(o, None)
    blocks = {"ovov": eri[O, V, O, V], "oovv": eri[O, O, V, V], "ovvo": eri[O, V, V, O], "ovvv": eri[O, V, V, V],
              "ovoo": eri[O, V, O, O], "oooo": eri[O, O, O, O], "vvvv": None if chol else eri[V, V, V, V]}
    rng = np.random.default_rng(seed)
    t1 = rng.standard_normal((o, v)) * 1e-2
    t2 = rng.standard_normal((o, o, v, v)) * 1e-2
    t2 = t2 + t2.transpose(1, 0, 3, 2)
    with gpu.Context(0) as ctx:
        ctx.set_ccsd_inputs(o, v, e, blocks, chol_vv=np.asfortranarray(L[:, o:, o:].transpose(1, 2, 0)) if chol else None)
        g1, g2 = ctx.ccsd_update(t1, t2)
    eia, eijab = co.denominators(e, o)
    r1, r2 = co.update_amplitudes(co.make_blocks(eri, o), eia, eijab, None, t1, t2)
    assert np.abs(g1 - r1).max() <= 1e-11 * np.abs(r1).max()
    assert np.abs(g2 - r2).max() <= 1e-11 * np.abs(r2).max()
