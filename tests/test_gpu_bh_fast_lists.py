"""The octree's fast mode where its term lists are short, ragged or full: the body counts at the edges
of a wave (one walks 64 bodies), of a list of 64 terms and of the 192 handed over at a time; groups of
one body; buckets longer than a list.

With theta = 0 every node is opened, so the force is the direct sum.  Bodies sit on a jittered unit
lattice, so a term's relative FP32 error is at most 3 * 2^-24 * (2 L / 0.5) (coordinates about the
group's centre against the smallest distance, cubed) plus a few 2^-24 and the sums' 64 * 2^-24: with
L <= 12 below 2e-5 of the sum of the terms' sizes.  A lost or doubled term is above 1e-3 of it."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 3, 63, 64, 65, 127, 128, 192, 193, 255, 257, 449, 1000])
@pytest.mark.parametrize("depth", [21, 1], ids=["tree", "buckets"])
def test_fast_lists_hold_every_term_once(oracle, n, depth):
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    ids = np.arange(n)
    b = gen.plummer(n, seed=1)
    for q, v in zip((b.x, b.y, b.z), (ids % side, ids // side % side, ids // side ** 2)):
        q[:] = v + rng.uniform(-0.25, 0.25, n)
    with NBodyGPU(G=1.0, precision="fp64", collisions=False) as g:
        g.load(b)
        g.bh_enable(theta=0.0, max_depth=depth, mode="fast")
        f, s = g.forces(), g.bh_stats()
    p = np.stack([b.x, b.y, b.z], 1)
    r3 = (((p[None] - p[:, None]) ** 2).sum(2) + 1e-8) ** 1.5
    size = (b.m[:, None] * b.m[None] * np.linalg.norm(p[None] - p[:, None], axis=2) / r3).sum(1)
    ref = oracle.force_soft(oracle.State.from_bodies(b), 1.0, 1e-4, nthreads=8)
    assert s["interactions"] == n * n and s["overflow"] == 0
    assert np.all(np.linalg.norm(f - ref, axis=1) <= 2e-5 * size)
