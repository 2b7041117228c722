"""The octree's build where its parts meet: body counts at the edges of a thread's four bodies, of a
block of 1,024 whose nodes one workgroup sums (and which counts nodes); a tight clump
across a block's end, so that deep nodes cross it; depth limits that make buckets.  Against the
host's insertion-built tree: leaf depths, node and bucket counts and, with theta = 0, the forces'
bits; with theta = 0.3 the forces to 1e-11 (the bar of the larger scenes: centres of mass are summed
from children, not body by body)."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 3, 4, 5, 8, 511, 512, 513, 1023, 1024, 1025, 1536, 2049, 5000])
@pytest.mark.parametrize("max_depth", [21, 4, 1])
@pytest.mark.parametrize("clump", [False, True])
def test_build_matches_insertion(oracle, n, max_depth, clump):
    rng = np.random.default_rng(n + max_depth)
    b = gen.plummer(n, seed=n)
    if clump:  # a third of the bodies within 1e-4 of one of them
        k = rng.choice(n, max(2, n // 3), replace=False)
        for q in (b.x, b.y, b.z):
            q[k] = q[k[0]] + rng.normal(0, 1e-4, len(k))
    st = oracle.State.from_bodies(b)
    for theta in (0.0, 0.3):
        with NBodyGPU(G=1.0, precision="fp64", collisions=False) as g:
            g.load(b)
            g.bh_enable(theta=theta, max_depth=max_depth)
            f, depth, s = g.forces(), g.bh_depths(), g.bh_stats()
        fo, do, info = oracle.bh_force(st, G=1.0, theta=theta, max_depth=max_depth)
        np.testing.assert_array_equal(depth, do)
        assert s["nodes"] - s["buckets"] == info["internal"]
        assert s["buckets"] == info["buckets"] and s["overflow"] == 0
        assert s["depth_max"] == info["max_depth_seen"]
        if theta == 0.0:
            np.testing.assert_array_equal(f, fo)
        else:
            d = np.linalg.norm(f - fo, axis=1) / np.linalg.norm(fo, axis=1)
            assert d.max() <= 1e-11
