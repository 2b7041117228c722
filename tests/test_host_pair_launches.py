"""Which launches the pair list takes: one workgroup's only where few pairs are known to be there, also
within a call of many cycles."""
import pytest

import host_only

SETUP = """
def per_cycle():
    out, cur = [], None
    for k in launched():
        if "k_zero_counters" in k:
            cur = []
            out.append(cur)
        elif cur is not None and "k_pair" in k:
            cur.append("small" if "k_pairs_small" in k else "wide")
    return ["small" if "small" in c else "wide" for c in out]

g = NBodyGPU(collisions=True)
b = gen.uniform_sphere(%d, 1)
g.load(b)
"""


@pytest.mark.parametrize("n,first", [(300, "small"), (4096, "small"), (4097, "wide"),
                                     (16384, "wide")])
def test_many_cycles_after_a_load(n, first):
    rc, out = host_only.run(SETUP % n + "first = %r" % first + """
fake.fake_pairs(60000)
fake.fake_clear()
g.step(1e-3, 1.0, nsteps=40)
assert per_cycle() == [first] + ["wide"] * 39, per_cycle()
fake.fake_pairs(100)                    # few: from the second cycle of the load's first call on
g.load(b)
fake.fake_clear()
g.step(1e-3, 1.0, nsteps=5)
assert per_cycle() == [first] + ["small"] * 4, per_cycle()
fake.fake_clear()
g.step(1e-3, 1.0, nsteps=3)
assert per_cycle() == ["small"] * 3, per_cycle()
fake.fake_pairs(5000)                   # the scene contracts during a call
fake.fake_clear()
g.step(1e-3, 1.0, nsteps=70)
assert per_cycle() == ["small"] * 32 + ["wide"] * 38, per_cycle()
print("done")
""")
    assert rc == 0 and "done" in out, (rc, out)


def test_room_for_many_pairs_in_a_small_scene():
    rc, out = host_only.run(SETUP % 1000 + """
g = NBodyGPU(collisions=True, pair_capacity=500000)
g.load(b)
fake.fake_clear()
g.step(1e-3, 1.0)
assert per_cycle() == ["wide"], per_cycle()
print("done")
""")
    assert rc == 0 and "done" in out, (rc, out)


def test_forces_after_a_load():
    rc, out = host_only.run(SETUP % 1000 + """
fake.fake_clear()
g.forces()
assert any("k_pair_rank" in k for k in launched()), launched()
assert not any("k_pairs_small" in k for k in launched())
print("done")
""")
    assert rc == 0 and "done" in out, (rc, out)
