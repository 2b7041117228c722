"""Pair lists of bodies that overlap very many others: put in order by bits, a window of 1,048,576
bodies at a time (nb_cycle.hip, k_pair_long)."""
import time

import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen

pytestmark = pytest.mark.gpu


def _hubs(n, seed, hubs):
    """Points that touch nothing, but for the given bodies, which reach all."""
    b = gen.plummer(n, seed)
    b.r[:] = 0.0
    b.r[hubs] = 100.0 * np.abs(b.pos()).max()
    return b


def _expected(n, hubs):
    i = np.arange(n)
    p = np.concatenate([np.stack([np.minimum(i, h), np.maximum(i, h)], 1)[i != h] for h in hubs])
    p = np.unique(p, axis=0)  # (two hubs meet once)
    return p.astype(np.int32)


# lists of 512 (in place), 513 and more; ends of the bit blocks; the second window
@pytest.mark.parametrize("n,hubs", [(9000, [512, 8999 - 513]), (16384, [0]), (16640, [16639]),
                                    (30001, [0, 1, 255, 256, 30000]), (1100000, [600000])])
def test_hub_lists(n, hubs):
    b = _hubs(n, 3, hubs)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, pair_capacity=8 * n) as g:
        g.load(b)
        for _ in range(2):
            g.forces()
            np.testing.assert_array_equal(g.pairs(), _expected(n, hubs))


@pytest.mark.parametrize("n", [700, 2000])
def test_all_overlap(n):
    b = gen.plummer(n, 5)
    b.r[:] = 100.0 * np.abs(b.pos()).max()
    i, j = np.triu_indices(n, 1)
    exp = np.stack([i, j], 1).astype(np.int32)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, pair_capacity=n * n // 2) as g:
        g.load(b)
        g.forces()
        np.testing.assert_array_equal(g.pairs(), exp)
        best = 1.0
        for _ in range(5):
            t = time.perf_counter()
            g.forces()
            best = min(best, time.perf_counter() - t)
        # 2 million pairs in lists of up to 1,999: 12 ms when a rank cost its list's length
        assert best < 6e-3, best
        np.testing.assert_array_equal(g.pairs(), exp)
