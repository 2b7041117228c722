"""The FP64 force in the reference's operation order, bit for bit against the oracle, at the sizes
at which the targets per workgroup change (4, 8, 16, 32, 64 lanes) and at the edges of their source
rounds (multiples of 13 * 64 / lanes): removed bodies, zero masses, bodies that share a coordinate
(zero numerators), and magnitudes that leave the shared reciprocal's range."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen

pytestmark = pytest.mark.gpu

NT = 16
G_REF = 6.673e-11


@pytest.mark.parametrize("n", [1, 2, 13, 207, 208, 209, 1000, 1025, 2049, 4097, 8193, 15000])
@pytest.mark.parametrize("mode", ["reference", "softened", "softened, gate"])
def test_bits(oracle, n, mode):
    b = gen.uniform_sphere(max(n, 2), seed=n, radius_k=0.08)
    if n == 1:
        b = type(b)(*(getattr(b, k)[:1] for k in ("x", "y", "z", "vx", "vy", "vz", "m", "r",
                                                  "beh", "flags", "rest", "frag", "fstep")))
    b.flags[3::17] = 0
    b.m[4::19] = 0.0
    b.x[5::7] = b.x[0]
    b.y[6::11] = b.y[0]
    st = oracle.State.from_bodies(b)
    if mode == "reference":
        kw, exp = {}, oracle.force_ref(st, G_REF, nthreads=NT)
    else:
        gate = mode.endswith("gate")
        kw = dict(eps=30.0, overlap_cutoff=gate)
        exp = oracle.force_soft(st, G_REF, 30.0, cutoff=gate, nthreads=NT)
    with NBodyGPU(precision="fp64", pair_capacity=1 << 20, **kw) as g:
        g.load(b)
        f = g.forces()
        pairs = g.pairs()
    act = b.active()
    np.testing.assert_array_equal(f[act], exp[act])
    assert not f[~act].any()
    np.testing.assert_array_equal(pairs, oracle.detect(st))


@pytest.mark.parametrize("scale", [1e-70, 1e45, 1e130])
def test_bits_outside_the_shared_range(oracle, scale):
    b = gen.uniform_sphere(700, seed=3, radius_k=0.01)
    for k in ("x", "y", "z", "r"):
        getattr(b, k)[:] *= scale
    b.m[::2] *= 1e-150
    st = oracle.State.from_bodies(b)
    with NBodyGPU(precision="fp64") as g:
        g.load(b)
        np.testing.assert_array_equal(g.forces(), oracle.force_ref(st, G_REF, nthreads=NT))
