"""Calls made while the interpreter ends (an atexit handler that saves a run)."""
import pytest

import host_only


@pytest.mark.parametrize("n", [1000, 200001])  # copies one after another; beside the read-back
def test_batch_store_in_an_exit_handler(n):
    rc, out = host_only.run("""
    import atexit
    b = gen.plummer(%d, 1)
    b.frag[:] = np.arange(b.n)
    g = NBodyBatch(G=1.0, eps=0.01)
    g.load([b])

    def save():
        got = g.store()
        for k in ("m", "r", "beh", "rest", "frag", "fstep"):
            np.testing.assert_array_equal(getattr(got, k), getattr(b, k))
            assert getattr(got, k) is not getattr(b, k)
        print("saved")

    atexit.register(save)
    """ % n)
    assert rc == 0 and "saved" in out, (rc, out)


def test_batch_store_without_threads():
    rc, out = host_only.run("""
    import threading
    g = NBodyBatch(G=1.0, eps=0.01)
    g.load([gen.plummer(200001, 1)])

    def none(self):
        raise RuntimeError("can't start new thread")

    threading.Thread.start = none
    assert g.store().n == 200001
    print("done")
    """)
    assert rc == 0 and "done" in out, (rc, out)
