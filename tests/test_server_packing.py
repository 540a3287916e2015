"""Ready requests of small simulations share one launch of their pair kernel,
the pair-symmetric kernels included, and the counters say so.  Launches are
counted on a host-memory runtime."""
import pytest

import fake_hip

# 16 simulations are resident; while the only stream is busy with one of them
# the others' requests queue up, and the next issue finds all 15 ready
WAVE = """
srv = steps.Server(streams=1, pack_max_n=PACK)
ids = []
for s in range(16):
    d, keep = make(s)
    ids.append(srv.add_sim(d, *cloud(N, L)))
for t in [srv.submit(i, steps.REQ_FORCE, PREC) for i in ids]:
    assert srv.wait(t).status == 0
import time
before = srv.stats()
fake.fake_set_busy(1)
fake.fake_reset_launches()
first = srv.submit(ids[0], steps.REQ_FORCE, PREC)
while launches(KERNEL) == 0:                        # it holds the stream from here on
    time.sleep(1e-3)
rest = [srv.submit(i, steps.REQ_FORCE, PREC) for i in ids[1:]]
fake.fake_set_busy(0)
for t in [first] + rest:
    assert srv.wait(t).status == 0
st = srv.stats()
print(launches(KERNEL) - 1, st["packed_launches"] - before["packed_launches"],
      st["packed_requests"] - before["packed_requests"])
srv.close()
"""

R3 = """
L = None
make = lambda s: steps.make_desc(steps.TOPO_R3)
"""
T3 = """
L = 100.0
make = lambda s: steps.make_desc(steps.TOPO_T3, is_periodic=1, L=L)
"""
S1R2 = """
L = 100.0
nr, nz = 24, 16
rho, z = np.arange(nr)[:, None] * (2.25 * 80.0 / (nr - 1)), (np.arange(nz)[None, :] + 0.5) * (L / nz) - 0.5 * L
tab = np.ascontiguousarray(np.stack([1e-6 * rho + 0 * z, 1e-6 * z + 0 * rho], axis=-1).reshape(-1))
make = lambda s: steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, s1r2_lookup=1, interp_order=2,
                                 s1r2_table=tab, s1r2_shape=(nr, nz))
"""
EWALD = """
L = 100.0
g = (np.arange(8) - 3.5) * (L / 8)
X, Y, Z = np.meshgrid(g, g, g, indexing="ij")
tab = np.ascontiguousarray(np.stack([X, Y, Z], axis=-1).reshape(-1)) * 1e-6
make = lambda s: steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=tab)
"""


def wave(tmp_path, setup, n, kernel, prec=0, pack=65536):
    # graphs off: a captured launch is not counted
    script = setup + f"N, PREC, PACK, KERNEL = {n}, {prec}, {pack}, {kernel!r}\n" + WAVE
    return [int(v) for v in fake_hip.run(tmp_path, script.replace("streams=1,", "streams=1, use_graphs=False,"))[0].split()]


@pytest.mark.parametrize("setup,n,kernel,prec", [
    (R3, 3000, "pair_kernel", 0), (R3, 9000, "sym_kernel", 0), (R3, 14400, "sym_mixed_kernel", 1),
    (T3, 9261, "sym_kernel", 0), (S1R2, 1536, "sym_s1r2_kernel", 0), (S1R2, 1536, "sym_s1r2_kernel", 1),
    (EWALD, 216, "sym_t3_kernel", 0), (EWALD, 729, "sym_t3_kernel", 1),
], ids=["r3-3000", "r3-9000", "r3-mixed-14400", "t3-9261", "s1r2-1536", "s1r2-mixed-1536", "ewald-216",
        "ewald-mixed-729"])
def test_one_launch_for_a_wave(tmp_path, setup, n, kernel, prec):
    assert wave(tmp_path, setup, n, kernel, prec) == [1, 1, 15]


def test_no_packing_when_it_is_off(tmp_path):
    assert wave(tmp_path, T3, 9261, "sym_kernel", pack=0) == [15, 0, 0]


def test_kernels_of_a_group_are_counted_by_themselves(tmp_path):
    """One variant and precision, two kernels (particles of one mass or not):
    a launch for each."""
    script = T3 + "N, PREC, PACK, KERNEL = 9261, 0, 65536, 'sym_kernel'\n" + WAVE.replace(
        "ids.append(srv.add_sim(d, *cloud(N, L)))",
        "x, M, h = cloud(N, L)\n    ids.append(srv.add_sim(d, x, M if s % 3 else 1.0 + np.arange(N), h))")
    out = fake_hip.run(tmp_path, script.replace("streams=1,", "streams=1, use_graphs=False,"))
    assert [int(v) for v in out[0].split()] == [2, 2, 15]
