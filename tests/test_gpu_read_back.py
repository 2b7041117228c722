"""Reading arrays back through the pinned staging: sizes around its single-thread limit (1 MiB in
all), its pieces (1 MiB), slices (4 MiB, 16 pieces) and its whole buffer (32 MiB), odd counts (byte
arrays that end inside a word), and contexts read by several threads at once."""
import threading

import numpy as np
import pytest

from nbodygo_amd import NBodyBatch, NBodyGPU, gen

pytestmark = pytest.mark.gpu


def scene(n, seed):
    rng = np.random.default_rng(seed)
    b = gen.plummer(max(n, 1), seed)
    b.flags[:] = rng.integers(0, 16, b.n).astype(np.uint8)
    b.beh[:] = rng.integers(0, 4, b.n)
    b.rest[:] = rng.random(b.n)
    b.frag[:] = rng.random(b.n)
    b.r[:] = rng.random(b.n)
    return b


def same(b, s):
    for k in ("x", "y", "z", "vx", "vy", "vz", "m", "r", "beh", "flags", "rest", "frag"):
        np.testing.assert_array_equal(getattr(s, k), getattr(b, k), err_msg=k)


@pytest.mark.parametrize("n", [1, 3, 257, 11270, 11275, 45001, 131071, 131073, 400003])
def test_store_and_render(n):
    b = scene(n, n)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False) as g:
        g.load(b)
        same(b, g.store())
        xyz, ex = g.render()
    e = (b.flags & 1).astype(bool)
    np.testing.assert_array_equal(ex, e.astype(np.uint8))
    np.testing.assert_array_equal(xyz, np.where(e[:, None], b.pos().astype(np.float32), 0))


def test_threads():
    """Four contexts, one thread each, reading at the same time."""
    scenes = [scene(n, n) for n in (50001, 90001, 1001, 120001)]
    bad = []

    def run(b):
        try:
            with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False) as g:
                g.load(b)
                for _ in range(10):
                    same(b, g.store())
        except BaseException as e:  # an assertion in a thread is reported below
            bad.append(e)

    ts = [threading.Thread(target=run, args=(b,)) for b in scenes]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


@pytest.mark.parametrize("sizes", [[1], [64, 1, 63, 65], [5000, 0, 300, 8191], [1] * 700,
                                   [220000, 7]])
def test_batch_store(sizes):
    sims = [gen.plummer(max(n, 1), k) for k, n in enumerate(sizes)]
    for k, n in enumerate(sizes):
        if n == 0:
            s = sims[k]
            sims[k] = type(s)(*(getattr(s, q)[:0] for q in ("x", "y", "z", "vx", "vy", "vz", "m",
                                                            "r", "beh", "flags", "rest", "frag",
                                                            "fstep")))
    with NBodyBatch() as bt:
        bt.load(sims)
        s = bt.store()
    same(gen.concat(*sims), s)
