"""The FP64 pass over flagged tiles takes its records three at a time, neighbouring records sharing the
sources they load.  Scenes with few and many overlapping pairs, so that the record counts leave every
remainder and records with short lists stand beside records with a whole slice; with and without
softening (one square root or two a test).  Bodies sit on a lattice of spacing 100 with jitter 20 and
radius 1; a partner is within the sum of the radii of every k-th body.

Forces against the oracle's gated FP64 sum: a term's relative FP32 error is at most about
3 * 2^-24 * (2 * 2000 / 50) (positions up to 2,000 against distances of 50 or more) = 1.5e-5 of its
size; partners are apart by less than the gate, so they add no term.  Pairs exactly."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen


@pytest.mark.gpu
@pytest.mark.parametrize("n,every", [(2, 1), (3, 2), (65, 64), (130, 40), (700, 100), (1500, 7),
                                     (1500, 2), (4097, 2)])
@pytest.mark.parametrize("eps", [0.0, 0.5])
def test_flagged_records_in_groups(oracle, n, every, eps):
    rng = np.random.default_rng(n + every)
    b = gen.plummer(n, seed=1, radius=1.0)
    side = int(np.ceil(n ** (1 / 3)))
    ids = np.arange(n)
    p = np.stack([ids % side, ids // side % side, ids // side ** 2], 1) * 100.0
    p += rng.uniform(-20, 20, p.shape)
    first = np.arange(0, n - 1, every + 1 if every > 1 else 2)
    step = rng.normal(size=(len(first), 3))
    p[first + 1] = p[first] + step / np.linalg.norm(step, axis=1)[:, None] * rng.uniform(
        0.5, 1.9, len(first))[:, None]
    p = rng.permutation(p)
    b.x[:], b.y[:], b.z[:] = p.T
    b.r[:] = 1.0
    st = oracle.State.from_bodies(b)
    ref = oracle.force_soft(st, 1.0, eps, cutoff=True, nthreads=8)
    with NBodyGPU(G=1.0, eps=eps, overlap_cutoff=True, collisions=True) as g:
        g.load(b)
        f, pairs = g.forces(), g.pairs()
    d = np.linalg.norm(p[None] - p[:, None], axis=2)
    near = d <= 2.0
    want = np.argwhere(np.triu(near, 1))
    np.testing.assert_array_equal(np.asarray(pairs).reshape(-1, 2), want)
    size = np.where(near, 0, b.m[:, None] * b.m[None] * d / (d * d + eps * eps) ** 1.5
                    if eps else b.m[:, None] * b.m[None] / np.where(near, 1, d) ** 2).sum(1)
    assert np.all(np.linalg.norm(f - ref, axis=1) <= 1.5e-5 * size + 1e-300)
