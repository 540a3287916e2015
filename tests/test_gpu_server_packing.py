"""Packed pair-symmetric launches: every simulation of a batch has the forces,
positions and velocities it has alone, to the bit, for each kernel the batch
may hold, several kernels and sizes in one batch included."""
import numpy as np
import pytest

import steps_amd
from steps_amd import workloads as wl

pytestmark = pytest.mark.gpu

L = 100.0
SP = steps_amd.StepParams(1e-4, 0.5, 100.0, 0.501, 99.0, 1.0, 1.0)


def cloud(N, seed, box=None, equal=False):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(N, 3)) * 30.0 if box is None else rng.uniform(0.0, box, (N, 3))
    M = np.full(N, 1.3) if equal else rng.uniform(0.5, 2.0, N)
    return x, M, np.full(N, 0.02), rng.normal(size=(N, 3))


def r3(steps):
    return [(steps.make_desc(steps.TOPO_R3), cloud(n, n, equal=e)) for n, e in
            ((700, 0), (8192, 0), (8193, 1), (14400, 0), (14401, 1), (20000, 0), (9000, 1), (3000, 0))]


def t3_nearest(steps):
    return [(steps.make_desc(steps.TOPO_T3, is_periodic=1, L=L), cloud(n, n, L, e)) for n, e in
            ((9261, 0), (9261, 1), (14500, 0), (14337, 1), (8200, 0), (1728, 0), (14600, 0), (14700, 1), (14800, 1))]


def s1r2_nearest(steps):
    return [(steps.make_desc(steps.TOPO_S1R2, is_periodic=1, L=L, Rsim=80.0), cloud(n, n, L, e))
            for n, e in ((8192, 0), (9001, 1), (10240, 0), (2000, 0), (8193, 0), (9002, 1), (8500, 1), (2001, 0), (2002, 0))]


def s1r2_table(order):
    def make(steps):
        T, shape = steps.s1r2_table(2, L, 80.0)
        return [(steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, s1r2_lookup=1, interp_order=order,
                                 s1r2_table=T, s1r2_shape=shape), cloud(n, n, L))
                for n in (1024, 1025, 1536, 3001, 900, 6000)]
    return make


def t3_ewald(steps):
    T = steps.t3_table(2, L)
    ng = round((T.size // 3) ** (1 / 3))
    g = (np.arange(8) - 3.5) * (L / 8)
    X, Y, Z = np.meshgrid(g, g, g, indexing="ij")
    small = np.ascontiguousarray(np.stack([X, Y, Z], axis=-1).reshape(-1)) * 1e-6
    bent = T.reshape(ng, ng, ng, 3).copy()
    bent[:, :, 40:, 2] *= 1.25                              # not odd: the one-sided kernel
    bent = bent.reshape(-1)
    return [(steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=t), cloud(n, n, L))
            for t, n in ((T, 216), (T, 729), (small, 700), (bent, 500), (T, 4096), (small, 9000), (bent, 700), (T, 130))]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("make", [r3, t3_nearest, s1r2_nearest, s1r2_table(2), s1r2_table(4), t3_ewald],
                         ids=["r3", "t3-nearest", "s1r2-nearest", "s1r2-cic", "s1r2-tsc", "t3-ewald"])
def test_batch_equals_alone(steps, make, precision):
    sims = make(steps)
    srv = steps_amd.Server(streams=1, use_graphs=False)
    ids = [srv.add_sim(d, x, M, h, v) for (d, keep), (x, M, h, v) in sims]
    print(f"case packed batch {[m[1][1].size for m in sims]} precision {precision}", flush=True)
    for t in [srv.submit(i, steps_amd.REQ_FORCE, precision) for i in ids]:  # resident from here on
        assert srv.wait(t).status == 0
    for _ in range(3):
        for t in [srv.submit(i, steps_amd.REQ_STEP, precision, SP) for i in ids]:
            assert srv.wait(t).status == 0
        for t in [srv.submit(i, steps_amd.REQ_FORCE, precision) for i in ids]:
            assert srv.wait(t).status == 0
    st = srv.stats()
    print(f"[packed batch] {st['packed_launches']} launches of {st['packed_requests']} requests", flush=True)
    # the first request of a wave may go alone; each kernel has three members or more
    assert st["packed_requests"] >= 2
    for i, ((d, keep), (x, M, h, v)) in zip(ids, sims):
        d.precision = precision
        sim = steps_amd.Sim(d, M.size)
        sim.set_state(x, M, h, v)
        sim.forces()
        for _ in range(3):
            sim.step(SP.h, SP.a_kick1, SP.hubble1, SP.a_kick2, SP.hubble2, SP.rho_part)
        sim.forces()
        xs, vs, F = srv.get_state(i)
        xa, va = sim.get_state()
        assert np.array_equal(F, sim.get_forces()) and np.array_equal(xs, xa) and np.array_equal(vs, va), M.size
        assert np.all(np.isfinite(F))
        sim.close()
        d.precision = 0
    srv.close()
