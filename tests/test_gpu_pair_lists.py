"""The pair list's canonical order and the chains built from it, where they can go wrong: a body
that overlaps thousands of others (one list with almost every pair), the body count at which the
whole pass leaves one workgroup's LDS (16,384), few pairs after many and many after few (the launches
follow the last cycle's count), no pair at all, and a list cut at its capacity."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, NBodyError, gen
from nbodygo_amd import _lib as L

pytestmark = pytest.mark.gpu


def hub_scene(n, seed, hubs):
    """Small bodies, and `hubs` large ones that each overlap a good part of the sphere."""
    b = gen.uniform_sphere(n, seed=seed, radius_k=0.002)
    at = np.linspace(0, n - 1, hubs).astype(int)
    b.r[at] = 300.0
    return b


@pytest.mark.parametrize("n,hubs", [(300, 1), (5000, 1), (16384, 2), (16385, 2)])
def test_long_lists_match_the_one_lane_pass(oracle, n, hubs):
    b = hub_scene(n, n, hubs)
    exp = oracle.detect(oracle.State.from_bodies(b))
    out = {}
    for resolve in (0, 1):
        with NBodyGPU(resolve=resolve, precision="fp64") as g:
            g.load(b)
            stats = [g.step(1e-3, 1.0) for _ in range(2)]
            out[resolve] = (g.store(), [s["resolved_total"] for s in stats], g.pairs())
            g.load(b)
            g.forces()
            np.testing.assert_array_equal(g.pairs(), exp)
    assert len(exp) > n // 200
    for k in ("x", "y", "z", "vx", "vy", "vz"):
        np.testing.assert_array_equal(getattr(out[0][0], k), getattr(out[1][0], k), err_msg=k)
    assert out[0][1] == out[1][1]
    np.testing.assert_array_equal(out[0][2], out[1][2])


def test_counts_follow_loads(oracle):
    """One context: 13,000 pairs, none, 100, 13,000 again; each list as the oracle's."""
    dense = gen.uniform_sphere(14000, seed=1, radius_k=0.05)
    none = gen.uniform_sphere(2000, seed=2, radius_k=0.0)
    few = gen.uniform_sphere(20000, seed=3, radius_k=0.01)
    with NBodyGPU() as g:
        for b in (dense, none, few, dense, few, none):
            g.load(b)
            g.forces()
            exp = oracle.detect(oracle.State.from_bodies(b))
            np.testing.assert_array_equal(g.pairs(), exp)
            s = g.step(1e-3, 1.0)
            assert s["pairs_total"] == len(exp)


def test_capacity(oracle):
    """A list cut at its capacity holds that many distinct pairs of the full list, in order."""
    b = gen.uniform_sphere(12000, seed=4, radius_k=0.05)
    full = {tuple(p) for p in oracle.detect(oracle.State.from_bodies(b))}
    with NBodyGPU(pair_capacity=1000) as g:
        g.load(b)
        with pytest.raises(NBodyError):
            g.forces()
        s = g.step(1e-3, 1.0, allow_overflow=True)
        assert s["pair_overflow"] == 1 and s["pairs_total"] == len(full)
        p = g.pairs()[:1000]  # (the call reports the whole count; the list holds its capacity)
    keys = p[:, 0].astype(np.int64) << 32 | p[:, 1]
    assert (np.diff(keys) > 0).all()
    assert all(tuple(q) in full for q in p)
    assert L.NB_E_PAIR_OVERFLOW == -4
