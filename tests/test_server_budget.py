"""The server's memory budget: an ensemble that fits with the least scratch
stays resident, with more scratch where there is room for it, and one that
does not takes turns.  On a host-memory runtime."""
import fake_hip

RUN = """
d, keep = steps.make_desc(steps.TOPO_R3)
N = 20000
probe = steps.Server(streams=1)
least = probe.sim_bytes(probe.add_sim(d, *cloud(N)))
probe.close()

def serve(count, budget, late=0):
    srv = steps.Server(streams=1, use_graphs=False, hbm_budget_bytes=budget)
    ids = [srv.add_sim(d, *cloud(N)) for _ in range(count)]
    most = 0
    for wave in range(3):
        if wave == 1:
            ids += [srv.add_sim(d, *cloud(N)) for _ in range(late)]
        for t in [srv.submit(i, steps.REQ_FORCE) for i in ids]:
            assert srv.wait(t).status == 0
            most = max(most, srv.stats()["bytes_resident"])
    st = srv.stats()
    srv.close()
    return st["resident_sims"], st["evictions"], most, st["admissions"]
"""


def serve(tmp_path, call):
    out = fake_hip.run(tmp_path, RUN + f"print(least, *serve({call}))\n")
    return [int(v) for v in out[0].split()]


def test_least_footprint(tmp_path):
    """Half as much again as state, tiles and the split sums of the one-sided
    kernel (52 in mixed precision), which a simulation took before the
    pair-symmetric slots, at the most."""
    least = serve(tmp_path, "1, 1 << 34")[0]
    assert least < 1.5 * 20000 * (112 + 24 * 52 + 160)


def test_ensemble_that_fits_stays_resident(tmp_path):
    least, resident, evictions, most, admissions = serve(tmp_path, "10, 10 * least")
    assert (resident, evictions, admissions) == (10, 0, 10) and most <= 10 * least


def test_room_that_is_left_is_used(tmp_path):
    least, resident, evictions, most, admissions = serve(tmp_path, "4, 1 << 34")
    assert (resident, evictions) == (4, 0) and most > 4 * least
    least, resident, evictions, most, admissions = serve(tmp_path, "10, 13 * least")
    assert (resident, evictions) == (10, 0) and 10 * least < most <= 13 * least


def test_simulations_added_later_get_their_room(tmp_path):
    """The first ones took the room; those that come later evict them once,
    and then all stay."""
    least, resident, evictions, most, admissions = serve(tmp_path, "3, 10 * least, late=7")
    assert resident == 10 and most <= 10 * least and evictions <= 3 and admissions == 10 + evictions


def test_ensemble_that_does_not_fit_takes_turns(tmp_path):
    least, resident, evictions, most, admissions = serve(tmp_path, "6, 3 * least")
    assert 1 <= resident < 6 and evictions > 0 and most <= 3 * least


def test_larger_than_the_budget(tmp_path):
    """A simulation alone above the budget takes less scratch than it is
    reported with, down to one cell; below that it is refused."""
    out = fake_hip.run(tmp_path, RUN + """
print(code(lambda: serve(1, least // 3)), *serve(1, least - 1), least)
""")
    rc, resident, evictions, most, admissions, least = [int(v) for v in out[0].split()]
    assert rc != 0 and resident == 1 and most < least


def test_small_simulation_in_a_small_budget(tmp_path):
    """N = 3000 takes 47 source splits where there is room; it needs the 11 of
    256 sources: 1.25 MB."""
    out = fake_hip.run(tmp_path, RUN + """
N = 3000
print(*serve(1, 1250000), code(lambda: serve(1, 1000000)))
""")
    resident, evictions, most, admissions, rc = [int(v) for v in out[0].split()]
    assert resident == 1 and most <= 1250000 and rc != 0
