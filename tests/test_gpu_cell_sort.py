"""The surrogate's sort of bodies by cell at the edges of its parts: a wave's 64 bodies, a workgroup's
1,024 (4,096 above 524,288 bodies), keys of up to 10 bits (one pass) and more (two), inactive bodies
last.  The same bodies in another order have the same cells: the counts of cells and of near pairs
agree exactly, the forces to FP32 rounding of sums in another order (a body lost, doubled or in a wrong
cell is above 1e-2 at these counts), and a repeated call gives the same bits."""
import numpy as np
import pytest

from nbodygo_amd import NBodyGPU, gen


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 4097, 20000, 530001])
@pytest.mark.parametrize("grid", [8, 10, 12, 64])
def test_order_of_the_bodies_does_not_matter(n, grid):
    if n > 20000 and grid != 64:
        pytest.skip("one size above 524,288 is enough")
    b = gen.plummer(n, seed=n)
    b.flags[::13] = 0
    b.flags[0] = 1
    p = np.random.default_rng(n).permutation(n)
    c = b.copy()
    for k in ("x", "y", "z", "m", "flags"):
        getattr(c, k)[:] = getattr(b, k)[p]
    out = []
    for s in (b, c):
        with NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False) as g:
            g.load(s)
            g.sur_enable(grid=grid, shell=2, r0=2.0, use_mlp=False, check_every=0)
            f = g.forces()
            st = g.sur_stats()
            np.testing.assert_array_equal(g.forces(), f)
        out.append((f, st["near_pairs_total"], st["nonempty_cells"]))
    assert out[0][1:] == out[1][1:]
    act = c.flags != 0  # (an inactive body's force is left as it was)
    f0, f1 = out[0][0][p][act], out[1][0][act]
    assert np.linalg.norm(f0 - f1) <= 1e-5 * np.linalg.norm(f0)
