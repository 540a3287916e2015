"""Where the scratch of a pair-symmetric or octree evaluation does not fit the
device, the call goes on with the least it can do with, and an allocation that
failed is not reported again by a later call.  On a host-memory runtime."""
import fake_hip

MAKE = """
d, keep = steps.make_desc(steps.TOPO_R3, **KW)
x, M, h = cloud(20000)
"""


def numbers(line):
    return [int(v) for v in line.split()]


def check(tmp_path, kw):
    out = fake_hip.run(tmp_path, f"KW = {kw}\n" + MAKE + """
sim = steps.Sim(d, 20000)
most = fake.fake_largest()
sim.close()
fake.fake_set_limit(most - 1)                       # the scratch is the largest piece
sim = steps.Sim(d, 20000)
print(most, fake.fake_largest())
print(code(lambda: sim.set_state(x, M, h)), code(sim.forces), code(sim.get_forces))
print(code(lambda: steps.force_eval(d, x, M, h)), fake.fake_largest())
fake.fake_set_limit(1 << 16)                        # nothing fits: refused ...
y, m, s = cloud(30000)
print(code(lambda: steps.force_eval(d, y, m, s)), code(lambda: steps.Sim(d, 30000)))
fake.fake_set_limit(NO_LIMIT)                       # ... and not the next calls
print(code(lambda: steps.force_eval(d, y, m, s)), code(lambda: steps.Sim(d, 30000)), code(sim.forces))
""")
    most, least = numbers(out[0])
    assert 0 < least < most
    assert numbers(out[1]) == [0, 0, 0]
    rc, used = numbers(out[2])
    assert rc == 0 and used < most
    refused = numbers(out[3])
    assert all(rc != 0 for rc in refused)
    assert numbers(out[4]) == [0, 0, 0]


def test_pair_symmetric(tmp_path):
    check(tmp_path, "dict()")


def test_octree(tmp_path):
    check(tmp_path, "dict(bh_theta=0.5, bh_particle_radius=0.1)")


def test_scratch_leaves_room_for_the_rest(tmp_path):
    """The scratch is taken after everything else a call or a simulation
    keeps: a device that holds it only without the rest runs with the least.
    A simulation that does not fit leaves nothing behind."""
    out = fake_hip.run(tmp_path, "KW = {}\n" + MAKE + """
sim = steps.Sim(d, 20000)
whole, most = fake.fake_live(), fake.fake_largest()
sim.close()
fake.fake_set_capacity(whole - 8)
sim = steps.Sim(d, 20000)
print(code(lambda: sim.set_state(x, M, h)), code(sim.forces), whole, fake.fake_live())
sim.close()
print(code(lambda: steps.force_eval(d, x, M, h)))
fake.fake_set_capacity(fake.fake_live() + 1000000)
before = fake.fake_live()
print(code(lambda: steps.Sim(d, 20000)), fake.fake_live() - before)
""")
    a, b, whole, now = numbers(out[0])
    assert a == 0 and b == 0 and now < whole
    assert numbers(out[1]) == [0]
    rc, left = numbers(out[2])
    assert rc != 0 and left == 0


def test_small_call_without_pinned_memory(tmp_path):
    out = fake_hip.run(tmp_path, "KW = {}\n" + """
d, keep = steps.make_desc(steps.TOPO_R3)
x, M, h = cloud(1500)
fake.fake_set_pinned_fails(1)
print(code(lambda: steps.force_eval(d, x, M, h)), code(lambda: steps.force_eval(d, x, M, h)))
fake.fake_set_pinned_fails(0)
print(code(lambda: steps.force_eval(d, x, M, h)))
""")
    assert numbers(out[0]) == [0, 0] and numbers(out[1]) == [0]
