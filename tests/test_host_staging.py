"""Copies and pinned memory of the read-backs: what a call asks of the runtime."""
import host_only


def test_a_network_alone_keeps_its_staging():
    rc, out = host_only.run("""
    from nbodygo_amd.mlp import MLP
    m = MLP(30, hidden=128, layers=8, d_out=3, seed=1)
    p = np.random.default_rng(1).standard_normal(m.n_params).astype(np.float32)
    m.set_params(p)
    before = fake.fake_host_mallocs()
    for _ in range(5):
        np.testing.assert_array_equal(m.get_params(), p)
        m.grad(np.zeros((64, 30), np.float32), np.zeros((64, 3), np.float32))
    assert fake.fake_host_mallocs() - before <= 1, fake.fake_host_mallocs()
    m.close()
    assert fake.fake_in_use() == 0
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)


def test_losses_of_a_layer_by_layer_step_are_written_where_they_are_kept():
    rc, out = host_only.run("""
    from nbodygo_amd.mlp import MLP
    x, t = np.zeros((256, 30), np.float32), np.zeros((256, 3), np.float32)
    m = MLP(30, hidden=128, layers=5, d_out=3, seed=1)
    for steps in (1, 10, 40):
        before = fake.fake_dev_copies()
        m.train(x, t, steps, batch=64)
        assert fake.fake_dev_copies() - before == steps   # the targets', once a step
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)
