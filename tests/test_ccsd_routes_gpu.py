"""One FP64 CCSD update at the sizes where its contractions change routes, against the oracle: 1e-11 of the largest
amplitude (FP64 sums in another order), as the other updates."""

import numpy as np
import pytest

from oracle import ccsd_oracle as co
from scess_amd import gpu
from scess_amd.synthetic import _draw, full_eri_chem

pytestmark = pytest.mark.gpu


def _check(o, v, seed):
    print(f"case ccsd routes o={o} v={v}", flush=True)
    e, L, _ = _draw(o, v, seed)
    L = L * 0.3
    eri = full_eri_chem(L)
    O, V = slice(0, o), slice(o, None)
    blocks = {"ovov": eri[O, V, O, V], "oovv": eri[O, O, V, V], "ovvo": eri[O, V, V, O], "ovvv": eri[O, V, V, V],
              "ovoo": eri[O, V, O, O], "oooo": eri[O, O, O, O]}
    rng = np.random.default_rng(seed)
    t1 = rng.standard_normal((o, v)) * 1e-2
    t2 = rng.standard_normal((o, o, v, v)) * 1e-2
    t2 = t2 + t2.transpose(1, 0, 3, 2)
    with gpu.Context(0) as ctx:
        ctx.set_ccsd_inputs(o, v, e, blocks, chol_vv=np.asfortranarray(L[:, o:, o:].transpose(1, 2, 0)))
        g1, g2 = ctx.ccsd_update(t1, t2)
    eia, eijab = co.denominators(e, o)
    r1, r2 = co.update_amplitudes(co.make_blocks(eri, o), eia, eijab, None, t1, t2)
    assert np.abs(g1 - r1).max() <= 1e-11 * np.abs(r1).max()
    assert np.abs(g2 - r2).max() <= 1e-11 * np.abs(r2).max()


# Foo and Fvv sum o v^2 (Fvv o^2 v) products per output: 16200 in one launch, 16562 as a split GEMM of 2 x 2 outputs
@pytest.mark.parametrize("o,v", [(2, 90), (2, 91)])
def test_long_sums(o, v):
    _check(o, v, v)


# Z = sum_cd (kd|ac) tau_ij^cd: (kd|ac) read in place as a batch over k with the sum over d, c split (96), permuted because
# its rows are too few per k (94) or not 16-byte aligned (97)
@pytest.mark.parametrize("o,v", [(4, 94), (4, 96), (4, 97)])
def test_operands_in_place(o, v):
    _check(o, v, v)
