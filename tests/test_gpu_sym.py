"""The force kernel that evaluates each unordered pair once (softened force, no overlap cutoff)
against the CPU FP64 oracle: sizes around its tiles (64), blocks (256, 512, 1,024) and the sizes at
which the targets per lane change (12,288 and 28,672), inactive bodies, detection, coordinates at
which the cube of 1/r leaves FP32's range, and a size whose block distances need two panels.

Tolerances are the FP32 path's: global 1e-5, per-body p99 1e-4; pair lists identical."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen
from nbodygo_amd import _lib as L

pytestmark = pytest.mark.gpu

NT = 16
SIZES = [1, 2, 63, 64, 65, 255, 257, 1000, 1024, 4097, 12287, 12288, 28671, 28672]


def errors(got, exp):
    norm = np.linalg.norm(exp)
    per = np.linalg.norm(got - exp, axis=1) / np.maximum(np.linalg.norm(exp, axis=1), 1e-300)
    return np.linalg.norm(got - exp) / (norm if norm > 0 else 1.0), np.percentile(per, 99)


@pytest.mark.parametrize("n", SIZES)
def test_forces_and_pairs(oracle, n):
    b = gen.plummer(max(n, 2), seed=n, radius=0.3 * max(n, 2) ** (-2.0 / 3.0))
    if n == 1:
        b = type(b)(*(getattr(b, k)[:1] for k in ("x", "y", "z", "vx", "vy", "vz", "m", "r",
                                                  "beh", "flags", "rest", "frag", "fstep")))
    b.flags[5::11] = 0                     # removed bodies: neither sources nor in a pair
    b.flags[7::13] |= L.NB_F_FRAGMENTING   # nor are fragmenting ones
    b.m[::3] *= 7.0
    st = oracle.State.from_bodies(b)
    idx = np.nonzero(b.active())[0]
    idx = idx[:: max(1, len(idx) // 1500)]
    exp = oracle.force_soft(st, 1.0, 0.01, idx=idx, nthreads=NT)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False) as g:
        g.load(b)
        assert g.config()["variant"] == 3
        f = g.forces()
        pairs = g.pairs()
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False) as g:
        g.load(b)
        np.testing.assert_array_equal(g.forces(), f)
    glob, p99 = errors(f[idx], exp)
    assert glob <= 1e-5 and p99 <= 1e-4
    np.testing.assert_array_equal(pairs, oracle.detect(st))


@pytest.mark.parametrize("n", [1000, 4097, 12288, 28672])
def test_pair_lists(oracle, n):
    """About n / 50 overlapping pairs (0.74 n^2 r^3 in a Plummer sphere), every behaviour."""
    b = gen.plummer(n, seed=n + 1, radius=0.3 * n ** (-1.0 / 3.0))
    b.beh[::7] = L.NB_CB_NONE
    b.beh[1::7] = L.NB_CB_FRAGMENT
    b.beh[2::7] = L.NB_CB_SUBSUME
    b.flags[5::11] = 0
    st = oracle.State.from_bodies(b)
    exp = oracle.detect(st)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False) as g:
        g.load(b)
        g.forces()
        np.testing.assert_array_equal(g.pairs(), exp)
    assert len(exp) > n // 500


@pytest.mark.parametrize("scale", [1e-9, 1e11, 1e13, 1e16])
def test_far_scales(oracle, scale):
    """Lengths times `scale`, masses times scale^3: the same accelerations times scale.  1 / r^3
    runs from 1e33 to 1e-48 over these; single precision's normal range ends at 1e-38."""
    b = gen.plummer(3000, seed=4)
    for k in ("x", "y", "z"):
        getattr(b, k)[:] *= scale
    b.m[:] *= min(scale, 1e12) ** 3
    st = oracle.State.from_bodies(b)
    exp = oracle.force_soft(st, 1.0, 0.01 * scale, nthreads=NT)
    with NBodyGPU(G=1.0, eps=0.01 * scale, overlap_cutoff=False, collisions=False) as g:
        g.load(b)
        f = g.forces()
    glob, p99 = errors(f / b.m[:, None], exp / b.m[:, None])
    assert glob <= 1e-5 and p99 <= 1e-4


def test_two_panels(oracle):
    """450,003 bodies: 220 block distances, more than the 1 GiB workspace holds at once."""
    b = gen.plummer(450003, seed=8)
    st = oracle.State.from_bodies(b)
    idx = np.sort(np.random.default_rng(2).choice(b.n, 256, replace=False))
    exp = oracle.force_soft(st, 1.0, 0.01, idx=idx, nthreads=NT)
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False) as g:
        g.load(b)
        f = g.forces()[idx]
        np.testing.assert_array_equal(g.forces()[idx], f)
    glob, p99 = errors(f, exp)
    assert glob <= 1e-5 and p99 <= 1e-4
