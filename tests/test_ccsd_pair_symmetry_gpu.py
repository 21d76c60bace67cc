"""CCSD with the Cholesky factor where t_ij^ab = t_ji^ba does not hold (a t2 of the caller, or an F12 driver): the terms
are then evaluated as the reference writes them. Against the oracle: 1e-11 of the largest amplitude for one update, as the
other updates; FP32 and BF16x3 products within 1e-4, as theirs."""

import numpy as np
import pytest

from oracle import ccsd_oracle as co
from scess_amd import gpu
from scess_amd.synthetic import _draw, full_eri_chem

pytestmark = pytest.mark.gpu


def _system(o, v, seed, scale):
    e, L, _ = _draw(o, v, seed)
    L = L * scale
    eri = full_eri_chem(L)
    O, V = slice(0, o), slice(o, None)
    blocks = {"ovov": eri[O, V, O, V], "oovv": eri[O, O, V, V], "ovvo": eri[O, V, V, O], "ovvv": eri[O, V, V, V],
              "ovoo": eri[O, V, O, O], "oooo": eri[O, O, O, O]}
    return e, eri, blocks, np.asfortranarray(L[:, o:, o:].transpose(1, 2, 0))


# compared on the host up to 65536 elements, on the device from there on (33-wide: the 32-wide tiles' edge); how far off:
# everywhere, or one element of the last tile
@pytest.mark.parametrize("o,v,seed,one", [(1, 5, 1, False), (3, 7, 2, False), (2, 33, 3, False), (4, 24, 4, True),
                                          (3, 65, 5, True), (8, 33, 6, False), (8, 33, 7, True), (4, 65, 8, True)])
def test_update_of_any_t2(o, v, seed, one):
    print(f"case ccsd any t2 o={o} v={v} one={one}", flush=True)
    e, eri, blocks, chol = _system(o, v, seed, 0.3)
    rng = np.random.default_rng(seed)
    t1 = rng.standard_normal((o, v)) * 1e-1
    t2 = rng.standard_normal((o, o, v, v)) * 1e-2
    if one:
        t2 = t2 + t2.transpose(1, 0, 3, 2)
        t2[0, o - 1, v - 1, v - 2] += 0.3
    ints = co.make_blocks(eri, o)
    eia, eijab = co.denominators(e, o)
    r1, r2 = co.update_amplitudes(ints, eia, eijab, None, t1, t2)
    with gpu.Context(0) as ctx:
        ctx.set_ccsd_inputs(o, v, e, blocks, chol_vv=chol)
        for prec, tol in (("fp64", 1e-11), ("fp32", 1e-4), ("bf16x3", 1e-4)):
            ctx.set_ccsd_precision(prec)
            g1, g2 = ctx.ccsd_update(t1, t2)
            assert np.abs(g1 - r1).max() <= tol * np.abs(r1).max(), prec
            assert np.abs(g2 - r2).max() <= tol * np.abs(r2).max(), prec


def test_solve_with_any_driver():
    o, v = 3, 6
    e, eri, blocks, chol = _system(o, v, 6, 0.3)
    rng = np.random.default_rng(1)
    f12 = {"residual": rng.standard_normal((o, o, v, v)) * 1e-2, "energy": rng.standard_normal((o, o, v, v)) * 1e-3}
    want = co.solve_rccsd_diis(eri, e, o, f12=f12)
    with gpu.Context(0) as ctx:
        ctx.set_ccsd_inputs(o, v, e, blocks, chol_vv=chol, t2_driver=f12["residual"], f12_energy=f12["energy"])
        r = ctx.ccsd_solve()
    assert r["converged"] and want["converged"]
    assert abs(r["E_CCSD"] - want["E_CCSD"]) < 1e-9
    assert np.abs(r["t2"] - want["t2"]).max() < 1e-7
