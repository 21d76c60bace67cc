"""BF16x3 W-build: tile edge 128 from v = 193 on. Every accumulator takes the same MFMAs in the same order whatever the
tile, so all F_ijk equal those of 64-wide tiles bit for bit."""

import numpy as np
import pytest

from scess_amd import gpu
from scess_amd.synthetic import make_triples_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("v", [192, 193, 208, 239])
def test_tiles_agree_bitwise(monkeypatch, v):
    print("case", v, flush=True)
    ctx = gpu.Context(0)
    ctx.set_triples_inputs(make_triples_inputs(3, v, v), ("bf16x3",))
    monkeypatch.delenv("SCESS_WBUILD_BLK", raising=False)
    E, F, _ = ctx.triples_forward("bf16x3", with_F=True)
    for blk in ("2", "4"):
        monkeypatch.setenv("SCESS_WBUILD_BLK", blk)
        e, f, _ = ctx.triples_forward("bf16x3", with_F=True)
        assert e == E and np.array_equal(f, F), blk
