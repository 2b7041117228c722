"""The batched force that takes each unordered pair once (the default until a shape is set), against
the FP64 softened direct sum of the oracle: simulation sizes around its tiles (64), blocks (256, 512,
1,024) and the sizes at which the targets per lane change (1,024 and 4,096), few simulations (which
get fewer targets per lane) and many, removed bodies, and the size above which the other kernel runs.

Tolerances are the FP32 path's: global 1e-5 per simulation."""
import numpy as np
import pytest

from nbodygo_amd import NBodyBatch, gen

pytestmark = pytest.mark.gpu

NT = 16


def check(oracle, sims, f):
    at = 0
    for s in sims:
        st = oracle.State.from_bodies(s)
        idx = np.nonzero(s.active())[0]
        idx = idx[:: max(1, len(idx) // 300)]
        exp = oracle.force_soft(st, 1.0, 0.01, idx=idx, nthreads=NT)
        got = f[at:at + s.n][idx]
        norm = np.linalg.norm(exp)
        assert np.linalg.norm(got - exp) <= 1e-5 * (norm if norm > 0 else 1.0), s.n
        at += s.n


@pytest.mark.parametrize("sizes", [[1, 2], [63, 64, 65], [255, 256, 257, 1023, 1024, 1025],
                                   [4095, 4096, 4097], [8192] * 3, [700] * 200,
                                   [5000, 300] * 60, [32768], [32769, 100]])
def test_sizes(oracle, sizes):
    sims = [gen.plummer(max(n, 2), seed=17 * k + n) for k, n in enumerate(sizes)]
    for k, n in enumerate(sizes):
        if n == 1:
            s = sims[k]
            sims[k] = type(s)(*(getattr(s, q)[:1] for q in ("x", "y", "z", "vx", "vy", "vz", "m",
                                                            "r", "beh", "flags", "rest", "frag",
                                                            "fstep")))
    for s in sims[::2]:
        s.flags[3::7] = 0
        s.m[1::3] *= 5.0
    with NBodyBatch(G=1.0, eps=0.01) as bt:
        bt.load(sims)
        f = bt.forces()
        np.testing.assert_array_equal(bt.forces(), f)  # whatever the queue's order
    check(oracle, sims, f)
