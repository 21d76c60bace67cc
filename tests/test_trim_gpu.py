"""scess_trim: the device memory that a context keeps for later calls goes back, and the next call is as before."""

import ctypes

import numpy as np
import pytest

from scess_amd import gpu

pytestmark = pytest.mark.gpu


def _free(ctx):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()  # of the runtime that the library is linked with
    assert ctx.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_trim_gives_memory_back():
    n = 70  # nao^4 doubles: 192 MB a tensor, two of them and more in one transform
    rng = np.random.default_rng(1)
    tei = np.asfortranarray(rng.standard_normal((n,) * 4))
    C = np.asfortranarray(rng.standard_normal((n, n)))
    with gpu.Context(0) as ctx:
        first = ctx.transform_tei(tei, C)
        before = _free(ctx)
        ctx.trim()
        after = _free(ctx)
        print("free", before, after, flush=True)
        assert after - before >= 2 * 8 * n ** 4
        ctx.trim()
        assert np.array_equal(ctx.transform_tei(tei, C), first)
