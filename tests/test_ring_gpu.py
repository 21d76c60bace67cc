"""Copies through the pinned ring: one context lives through the module and has copied the 64 MiB after which the ring is
made, so every copy of 4 MiB or more below goes through it (tests/test_buffers_cpu.py counts them on a simulated device)."""

import threading

import numpy as np
import pytest

from scess_amd import gpu

pytestmark = pytest.mark.gpu


def _tei(n, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal((n, n, n, n)))


@pytest.fixture(scope="module", autouse=True)
def ring():
    with gpu.Context(0) as ctx:
        g = _tei(49, 0)  # 46 MB
        for _ in range(2):
            assert np.array_equal(ctx.transform_tei(g, np.eye(49)), g)
        yield


# n^4 doubles: below 4 MiB, a little above (a last chunk of a few KiB), whole 2 MiB chunks (32: 8 MiB), fewer chunks than
# the ring's eight slots and more
@pytest.mark.parametrize("n", [26, 27, 28, 32, 33, 38, 41, 49])
def test_round_trip_is_exact(n):
    g = _tei(n, n)
    with gpu.Context(0) as ctx:  # the identity transform: products with 1 and sums with 0 leave every bit
        for _ in range(2):
            assert np.array_equal(ctx.transform_tei(g, np.eye(n)), g)


def test_threads_and_contexts():
    bad = []

    def work(seed):
        for rep in range(4):
            with gpu.Context(0) as ctx:
                g = _tei(36, 10 * seed + rep)
                for _ in range(2):
                    if not np.array_equal(ctx.transform_tei(g, np.eye(36)), g):
                        bad.append((seed, rep))

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
