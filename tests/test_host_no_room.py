"""Device memory that runs out: workspaces of the kernels that take each pair once are given up for
the kernels that need none, and the call succeeds as it did before there were such workspaces."""
import host_only


def test_a_context_without_room_for_the_workspace():
    rc, out = host_only.run("""
    n = 262144
    b = gen.plummer(n, 1)
    kw = dict(G=1.0, eps=0.01, overlap_cutoff=False, collisions=True)
    g = NBodyGPU(variant=2, **kw)
    g.load(b)
    need = fake.fake_in_use()           # one evaluation per ordered pair
    g.close()
    for room in (1 << 20, 100 << 20, 300 << 20, 1 << 30):
        fake.fake_budget(need + room)
        g = NBodyGPU(**kw)
        g.load(b)
        v = g.config()["variant"]
        assert v == (3 if room >= 1 << 30 else 2), (room, v)
        g.step(1e-3, 1.0)               # (no error left over from the failed allocation)
        fake.fake_budget(200 << 20)     # (cycle's second set)
        g.add_bodies(gen.plummer(5, 2))
        g.cycle(1.0)
        g.autotune(1)
        g.step(1e-3, 1.0)
        g.close()
        assert fake.fake_in_use() == 0
    fake.fake_budget(need + (300 << 20))
    g = NBodyGPU(variant=3, **kw)       # asked for: refused
    try:
        g.load(b)
        raise SystemExit("accepted")
    except L.NBodyError as e:
        assert e.code == L.NB_E_HIP, e
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)


def test_slices_of_very_many_bodies():
    """12,288 rows of 1,024 bodies: 8 slices of 24 bytes a body, not 12."""
    rc, out = host_only.run("""
    n = 12288 * 1024
    z = np.zeros(n)
    from nbodygo_amd import Bodies
    g = NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False)
    g.load(Bodies(z, z, z, z, z, z, z, z))
    c = g.config()
    assert c["variant"] == 3 and c["jsplit"] == 8, c
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)


BATCH = """
sims = [gen.plummer(4000 + k, k) for k in range(16)]
g = NBodyBatch(G=1.0, eps=0.01)
g.load(sims)
full = fake.fake_in_use()
g.step(1e-3, 1.0)
assert any("k_batch_sym" in k for k in launched())
g.close()
assert fake.fake_in_use() == 0
"""


def test_a_batch_without_room_for_the_workspace():
    rc, out = host_only.run(BATCH + """
fake.fake_clear()
fake.fake_budget(full - (1 << 20))
g = NBodyBatch(G=1.0, eps=0.01)
g.load(sims)
g.step(1e-3, 1.0)
assert any("k_batch_force" in k for k in launched())
assert not any("k_batch_sym" in k for k in launched())
g.load(sims[:4])                        # fewer: there is room again
g.step(1e-3, 1.0)
assert any("k_batch_sym" in k for k in launched())
g.close()
print("done")
""")
    assert rc == 0 and "done" in out, (rc, out)


def test_a_batch_read_back_without_room_to_reorder():
    rc, out = host_only.run(BATCH + """
sims = [gen.plummer(1 + 37 * (k % 9), k) for k in range(150)]
g = NBodyBatch(G=1.0, eps=0.01)
g.load(sims)
fake.fake_budget(1000)
got = g.store()
exp = gen.concat(*sims)
for k in ("x", "y", "z", "vx", "vy", "vz", "flags"):
    np.testing.assert_array_equal(getattr(got, k), getattr(exp, k))
g.step(1e-3, 1.0)
g.close()
print("done")
""")
    assert rc == 0 and "done" in out, (rc, out)


def test_training_without_room_for_the_two_launch_step():
    """Layer by layer, the losses read step by step: as much memory as before there were its buffers."""
    rc, out = host_only.run("""
    from nbodygo_amd.mlp import MLP
    B, steps = 1 << 20, 40
    x, t = np.zeros((B, 30), np.float32), np.zeros((B, 3), np.float32)
    m = MLP(30, hidden=128, layers=3, d_out=3, seed=1)
    m.grad(x, t)                                  # (the layer-by-layer buffers)
    m.train(x, t, steps, batch=B)
    assert sum("k_train_rows" in k for k in launched()) == steps
    m.close()
    for room in (0, 4 << 20):
        m = MLP(30, hidden=128, layers=3, d_out=3, seed=1)
        m.grad(x, t)
        fake.fake_clear()
        fake.fake_budget(B * 34 * 4 + room)       # rows, targets and one step's losses
        m.train(x, t, steps, batch=B)
        assert not any("k_train_rows" in k for k in launched())
        assert sum("k_adam" in k for k in launched()) == 8 * steps
        fake.fake_budget((1 << 64) - 1)
        fake.fake_clear()
        m.train(x, t, 3, batch=B)
        assert sum("k_train_rows" in k for k in launched()) == 3
        m.close()
    assert fake.fake_in_use() == 0
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)
