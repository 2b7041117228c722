"""Host memory that runs out inside a call of the C interface: an error code or success, never an
exception out of the call (which would end the process)."""
import pytest

import host_only

STORE = """
b = gen.plummer(%d, 1)
g = NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False)
g.load(b)
for k in range(60):
    fake.fake_fail_new(k)
    try:
        g.store()
        g.render()
    except L.NBodyError as e:
        assert e.code in (L.NB_E_HIP, L.NB_E_NOMEM), e
    if fake.fake_new_left() >= 0:
        break                     # fewer than k allocations: all of them have failed once
    fake.fake_fail_new(-1)
    g.store()
fake.fake_fail_new(-1)
g.close()
print("done", k)
"""


@pytest.mark.parametrize("n", [1000, 100000, 600000])  # one launch; threads; several windows
def test_read_back_without_host_memory(n):
    rc, out = host_only.run(STORE % n)
    assert rc == 0 and "done" in out, (rc, out)


def test_add_without_host_memory_leaves_the_queue_alone():
    rc, out = host_only.run("""
    g = NBodyGPU(G=1.0, eps=0.01, overlap_cutoff=False, collisions=False)
    g.load(gen.plummer(100, 1))
    a = gen.plummer(10, 2)
    failed = 0
    for k in range(40):
        fake.fake_fail_new(k)
        try:
            g.add_bodies(a)
        except L.NBodyError as e:
            assert e.code == L.NB_E_NOMEM, e
            failed += 1
        if fake.fake_new_left() >= 0:
            break
    fake.fake_fail_new(-1)
    n = g.cycle(1.0)              # (no kernel runs: nothing of the first 100 survives)
    assert failed >= 3 and n == 10 * (k + 1 - failed), (failed, k, n)
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)


def test_batch_load_without_host_memory():
    rc, out = host_only.run("""
    sims = [gen.plummer(300 + k, k) for k in range(8)]
    g = NBodyBatch(G=1.0, eps=0.01)
    loaded = failed = 0
    for k in range(200):
        fake.fake_fail_new(k)
        try:
            g.load(sims)
            loaded += 1
        except L.NBodyError as e:
            assert e.code == L.NB_E_NOMEM, e
            failed += 1
        if fake.fake_new_left() >= 0:
            break
    fake.fake_fail_new(-1)
    assert failed and loaded > 1, (failed, loaded)   # (without the pairs-once lists it still loads)
    g.load(sims)
    g.step(1e-3, 1.0)
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)


def test_training_without_host_memory():
    rc, out = host_only.run("""
    from nbodygo_amd.mlp import MLP
    x, t = np.zeros((256, 30), np.float32), np.zeros((256, 3), np.float32)
    m = MLP(30, hidden=64, layers=2, d_out=3, seed=1)
    for k in range(20):
        fake.fake_fail_new(k)
        try:
            m.train(x, t, 50, batch=64)
        except L.NBodyError as e:
            assert e.code == L.NB_E_NOMEM, e
        if fake.fake_new_left() >= 0:
            break
        if k == 0:
            m.close()
            m = MLP(30, hidden=64, layers=2, d_out=3, seed=1)
    print("done", k)
    """)
    assert rc == 0 and "done" in out, (rc, out)
