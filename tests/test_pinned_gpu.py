"""Host arrays that the caller has pinned: copied directly, bit for bit, also once the copy ring is there."""

import ctypes

import numpy as np
import pytest

from scess_amd import gpu

pytestmark = pytest.mark.gpu


def _pinned(lib, shape):
    p = ctypes.c_void_p()
    n = int(np.prod(shape))
    assert lib.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(8 * n), 0) == 0
    a = np.frombuffer((ctypes.c_double * n).from_address(p.value)).reshape(shape, order="F")
    return p, a


def test_pinned_arrays():
    n = 49  # 46 MB
    g = np.asfortranarray(np.random.default_rng(n).standard_normal((n,) * 4))
    one = np.eye(n)
    with gpu.Context(0) as ctx:
        assert np.array_equal(ctx.transform_tei(g, one), g)  # 92 MB: the ring is made
        p, x = _pinned(ctx.lib, g.shape)
        q, y = _pinned(ctx.lib, g.shape)
        try:
            x[...] = g
            for _ in range(2):
                y[...] = 0.0
                ctx.check(ctx.lib.scess_transform_tei(ctx.h, n, n, gpu._ptr(x), gpu._ptr(one), 0, gpu._ptr(y)))
                assert np.array_equal(y, g)
        finally:
            assert ctx.lib.hipHostFree(p) == 0 and ctx.lib.hipHostFree(q) == 0
