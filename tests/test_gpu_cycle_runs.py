"""Compaction where its parts meet: body counts at the edges of the 256 bodies a workgroup takes at a
time and of its run of 1,024, everything or nothing removed, adds of none, one and many, with and
without the events' extra arrays.  Against the same done on the host: survivors in order, then the
queued bodies, last first, with the cycle's restitution.  Exact."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen
from nbodygo_amd import _lib as L

KEYS = ("x", "y", "z", "vx", "vy", "vz", "m", "r", "beh", "flags", "rest", "frag")


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 63, 256, 257, 1023, 1024, 1025, 2048, 5001])
@pytest.mark.parametrize("gone", [0.0, 0.3, 1.0])
@pytest.mark.parametrize("events", [False, True])
def test_survivors_and_adds_in_order(n, gone, events):
    rng = np.random.default_rng(n)
    b = gen.plummer(n, seed=n)
    b.rest[:] = rng.random(n)
    b.frag[:] = rng.random(n)
    b.flags[rng.random(n) < gone] = 0
    live = (b.flags & L.NB_F_EXISTS) != 0
    with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=events, events=events) as g:
        for nadd in (0, 1, 700):
            g.load(b)
            a = gen.plummer(max(nadd, 1), seed=n + 1)
            a.frag[:] = rng.random(a.n)
            if nadd:
                g.add_bodies(a)
            got_n = g.cycle(0.25)
            exp = {k: getattr(b, k)[live] for k in KEYS}
            if nadd:
                for k in KEYS:
                    v = np.full(nadd, 0.25) if k == "rest" else getattr(a, k)[::-1]
                    exp[k] = np.concatenate([exp[k], v])
            assert got_n == len(exp["x"])
            s = g.store()
            for k in KEYS:
                np.testing.assert_array_equal(getattr(s, k), exp[k], err_msg=k)
            # the new set steps like a fresh load of the same bodies
            assert g.step(0.0, nsteps=0)["n_active"] == got_n
