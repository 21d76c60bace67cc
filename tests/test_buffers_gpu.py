"""Copies between pageable host memory and the device through the pinned ring, and blocks reused between calls."""

import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tei(n, seed):
    return np.asfortranarray(np.random.default_rng(seed).standard_normal((n, n, n, n)))


# n^4 doubles: below the ring's 4 MiB, a little above, whole 2 MiB chunks (32: 8 MiB), more chunks than slots
@pytest.mark.parametrize("n", [3, 26, 27, 28, 32, 33, 41, 49])
def test_round_trip_is_exact(n):
    from scess_amd import gpu
    ctx = gpu.Context(0)
    g = _tei(n, n)
    # the identity transform: products with 1 and sums with 0 leave every bit
    for _ in range(2):
        assert np.array_equal(ctx.transform_tei(g, np.eye(n), chem_to_phys=False), g)


def test_two_threads_and_contexts():
    from scess_amd import gpu
    bad = []

    def work(seed):
        for rep in range(4):
            ctx = gpu.Context(0)
            g = _tei(36, 10 * seed + rep)
            for _ in range(2):
                if not np.array_equal(ctx.transform_tei(g, np.eye(36), chem_to_phys=False), g):
                    bad.append((seed, rep))
            del ctx

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_blocks_do_not_leak_between_inputs():
    """Gradients and energies of one context after larger and smaller inputs equal those of a fresh one."""
    from scess_amd import gpu, synthetic
    one = gpu.Context(0)
    for o, v in [(4, 30), (3, 9), (5, 41), (4, 30), (2, 17)]:
        x = synthetic.make_triples_inputs(o, v, seed=o + v)
        new = gpu.Context(0)
        got = []
        for ctx in (one, new):
            ctx.set_triples_inputs(x, ("fp64",))
            E, F, _ = ctx.triples_forward("fp64", with_F=True)
            got.append((E, F, ctx.triples_backward("fp64")))
        assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
        for k in got[1][2]:
            assert np.array_equal(got[0][2][k], got[1][2][k]), k
