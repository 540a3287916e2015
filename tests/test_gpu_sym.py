"""The pair-symmetric evaluation (every unordered pair once) against the CPU
oracle: block counts of both parities, a last block and a last tile that are
ragged, close and coincident pairs, row ranges it takes and leaves, and the
same sums whatever scratch it is given."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err, report
from steps_amd import _abi
from steps_amd import workloads as wl

pytestmark = pytest.mark.gpu

MIN_N = 8192          # sym_kernels.hip: the smallest N it takes


def particles(mode, N, seed):
    """Uniform particles with pairs inside the softening length and one
    coincident pair, in a box (T3, S1R2) or a ball-like cloud (R3)."""
    rng = np.random.default_rng(seed)
    L = 100.0
    x = rng.uniform(0.0, L, (N, 3))
    if mode == "r3":
        x = rng.normal(size=(N, 3)) * 30.0
    if mode == "s1r2":
        x[:, :2] = rng.normal(size=(N, 2)) * 60.0
    x[1:200:2] = x[0:199:2] + rng.normal(size=(100, 3)) * 0.02
    x[N - 1] = x[N - 2]                                   # coincident, in the ragged tile
    if mode != "r3":
        x[:, 2] %= L
    if mode == "t3":
        x %= L
    return x, rng.uniform(0.5, 2.0, N), np.full(N, 0.03), L


def descriptor(steps, oracle, mode, L):
    if mode == "r3":
        kw = dict(cosmology=1, comoving=1, mass_in_unit_sphere=0.7)
        return steps.make_desc(steps.TOPO_R3, **kw), oracle.params(0, **kw)
    if mode == "t3":
        return steps.make_desc(steps.TOPO_T3, is_periodic=1, L=L), oracle.params(1, is_periodic=1, L=L, interp_order=4)
    kw = dict(is_periodic=1, L=L, Rsim=300.0)
    return steps.make_desc(steps.TOPO_S1R2, **kw), oracle.params(2, cut_inclusive=0, **kw)


@pytest.mark.parametrize("N", [MIN_N, MIN_N + 1, 9 * 1024, 10 * 1024 - 63, 66001])
@pytest.mark.parametrize("mode", ["r3", "t3", "s1r2"])
def test_against_oracle(steps, oracle, mode, N):
    print(f"case pair-symmetric {mode} N={N}", flush=True)
    x, M, h, L = particles(mode, N, N)
    (d, keep), p = descriptor(steps, oracle, mode, L)
    F = steps.force_eval(d, x, M, h)
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(N - 40, N),
                                     np.linspace(0, N - 1, 60).astype(int)])).astype(np.int32)
    e = rel_err(F[rows], oracle.forces_rows(p, x, M, h, rows))
    report(f"pair-symmetric {mode} N={N}", e)
    # FP64 bars of every path: median 1e-12 (summation order), max 1e-10
    assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-10
    # most rows asked for: the same evaluation; few: the one-sided kernel
    assert np.array_equal(steps.force_eval(d, x, M, h, id_min=70, id_max=N - 2), F[70:N - 1])
    few = steps.force_eval(d, x, M, h, id_min=0, id_max=N // 2)
    assert np.median(rel_err(few, F[:N // 2 + 1])) <= 1e-12


@pytest.mark.parametrize("N", [12288, 12289, 14336, 15 * 1024 - 63, 66001])
@pytest.mark.parametrize("mode", ["r3", "t3", "s1r2"])
def test_mixed_against_fp64(steps, oracle, mode, N):
    """Mixed precision against FP64 on every row (the pair-sum bar, p99 1e-5),
    close pairs and pairs across the box edge included; deterministic."""
    print(f"case pair-symmetric mixed {mode} N={N}", flush=True)
    x, M, h, L = particles(mode, N, N)
    if mode != "r3":
        x[300:330, 2] = 1e-9 * np.arange(30)              # either side of the wrap
        x[330:360, 2] = L / 2 + 1e-8 * (np.arange(30) - 15)  # half a period away
    (d, keep), _ = descriptor(steps, oracle, mode, L)
    d.cosmology = 0
    F = steps.force_eval(d, x, M, h)
    d.precision = steps.PREC_MIXED
    Fm = steps.force_eval(d, x, M, h)
    e = rel_err(Fm, F)
    report(f"pair-symmetric mixed {mode} N={N} vs fp64", e)
    assert np.all(np.isfinite(Fm)) and np.median(e) <= 2e-6 and np.percentile(e, 99) <= 1e-5 and e.max() <= 1e-3
    assert not np.array_equal(Fm, F) and np.array_equal(steps.force_eval(d, x, M, h), Fm)


@pytest.mark.parametrize("N", [200, 256, 1087, 3000, 40001, 66000, 107001])
def test_t3_ewald_against_oracle(steps, oracle, N):
    """Every rows-per-workgroup choice of the T3 Ewald kernel (64, 128, 256
    by particles per table column), windows that fit and that do not, ragged
    ends, close pairs; and a table that is not odd through its centre, which
    has to take the one-sided kernel."""
    print(f"case pair-symmetric t3 ewald N={N}", flush=True)
    x, M, h, L = particles("t3", N, N)
    T = steps.t3_table(2, L)
    rows = np.unique(np.concatenate([np.arange(0, 12), np.arange(N - 12, N),
                                     np.linspace(0, N - 1, 24).astype(int)])).astype(np.int32)
    bent = T.reshape(63, 63, 63, 3).copy()
    bent[:, :, 40:, 2] *= 1.25                            # even in x and y still, not odd in z
    for label, tab in (("odd", T), ("bent", bent.reshape(-1))):
        if label == "bent" and N > 3000:
            continue
        d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=tab)
        F = steps.force_eval(d, x, M, h)
        p = oracle.params(1, is_periodic=2, L=L, t3_table=tab, interp_order=4)
        e = rel_err(F[rows], oracle.forces_rows(p, x, M, h, rows))
        report(f"pair-symmetric t3 ewald {label} N={N}", e)
        assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-9
        assert np.array_equal(steps.force_eval(d, x, M, h), F)
        dm, keepm = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=tab, precision=steps.PREC_MIXED)
        Fm = steps.force_eval(dm, x, M, h)
        em = rel_err(Fm, F)
        report(f"pair-symmetric t3 ewald {label} N={N} mixed vs fp64", em)
        # the mixed path's bar, p99 1e-5 (uniform particles, no cancelling lattice)
        assert np.all(np.isfinite(Fm)) and np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5
        assert not np.array_equal(Fm, F) and np.array_equal(steps.force_eval(dm, x, M, h), Fm)


@pytest.mark.parametrize("N", [1024, 1025, 5 * 256 - 63, 20011])
@pytest.mark.parametrize("order", [2, 4])
def test_s1r2_table_against_oracle(steps, oracle, order, N):
    """CIC and TSC, windows of rho rows that fit (particles sorted by radius)
    and that do not (shuffled), ragged ends and close pairs, both precisions;
    and a table that is not odd in z, which takes the one-sided kernel."""
    print(f"case pair-symmetric s1r2 order={order} N={N}", flush=True)
    x, M, h, L = particles("s1r2", N, N)
    Rsim = 300.0
    T, shape = steps.s1r2_table(2, L, Rsim)
    bent = T.reshape(*shape, 2).copy()
    bent[:, 3 * shape[1] // 4:, 1] *= 1.25
    by_radius = np.argsort(np.hypot(x[:, 0], x[:, 1]), kind="stable")
    rows = np.unique(np.concatenate([np.arange(0, 20), np.arange(N - 20, N),
                                     np.linspace(0, N - 1, 40).astype(int)])).astype(np.int32)
    for label, tab, o in (("by radius", T, by_radius), ("shuffled", T, np.arange(N)), ("bent", bent.reshape(-1), by_radius)):
        kw = dict(is_periodic=2, L=L, Rsim=Rsim, s1r2_lookup=1, interp_order=order, s1r2_table=tab, s1r2_shape=shape)
        d, keep = steps.make_desc(steps.TOPO_S1R2, **kw)
        dm, keepm = steps.make_desc(steps.TOPO_S1R2, precision=steps.PREC_MIXED, **kw)
        xo, Mo, ho = x[o], M[o], h[o]
        F = steps.force_eval(d, xo, Mo, ho)
        e = rel_err(F[rows], oracle.forces_rows(oracle.params(2, **kw), xo, Mo, ho, rows))
        report(f"pair-symmetric s1r2 order={order} N={N} {label}", e)
        assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-9
        Fm = steps.force_eval(dm, xo, Mo, ho)
        em = rel_err(Fm, F)
        report(f"pair-symmetric s1r2 order={order} N={N} {label} mixed vs fp64", em)
        # the mixed path's bar on the pair sum
        assert np.all(np.isfinite(Fm)) and np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5
        assert not np.array_equal(Fm, F)


@pytest.mark.parametrize("N", [150001, 300000])
def test_scratch_does_not_change_the_sums(steps, N):
    """The entry point with 256 MiB of static scratch runs fewer offsets a
    launch than the one that allocates: bitwise the same forces."""
    print(f"case pair-symmetric scratch N={N}", flush=True)
    w = wl.r3_compactified(N=N, seed=4)
    d, keep = steps.make_desc(steps.TOPO_R3, cosmology=1, comoving=1, mass_in_unit_sphere=w.mass_in_unit_sphere)
    F = steps.force_eval(d, w.x, w.M, w.soft)
    G = np.zeros(3 * N)
    lib = steps.load_library()
    x, M, h = (np.ascontiguousarray(a, dtype=np.float64) for a in (w.x.reshape(-1), w.M, w.soft))
    rc = lib.steps_force_eval_noalloc(C.byref(d), N, _abi._ptr(x), _abi._ptr(M), _abi._ptr(h), _abi._ptr(G), 0, N - 1)
    assert rc == 0, lib.steps_last_error()
    assert np.array_equal(G.reshape(-1, 3), F)


@pytest.mark.parametrize("ng", [3, 4, 8, 31, 62, 63])
@pytest.mark.parametrize("N", [700, 30011])
def test_t3_ewald_grids_against_oracle(steps, oracle, ng, N):
    """Tables of even and odd grids that are mirrored in x, y and z, which the
    window holds for z >= 0 only; pairs at dz = 0, at half a period and around."""
    print(f"case pair-symmetric t3 ewald ng={ng} N={N}", flush=True)
    x, M, h, L = particles("t3", N, N)
    x[400:460, 2] = 10.0 + 1e-13 * (np.arange(60) % 5)
    x[460:520, 2] = 10.0 + L / 2 + 1e-9 * (np.arange(60) - 30)
    x %= L
    g = (np.arange(ng) - (ng - 1) / 2) * (L / ng)
    X, Y, Z = np.meshgrid(g, g, g, indexing="ij")
    f = 1e-6 * np.exp(-(X * X + Y * Y + Z * Z) / (0.1 * L * L))
    T = np.ascontiguousarray(np.stack([X * f, Y * f, Z * f], axis=-1).reshape(-1))
    d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T)
    p = oracle.params(1, is_periodic=2, L=L, t3_table=T, interp_order=4)
    rows = np.unique(np.concatenate([np.arange(395, 525, 3), np.linspace(0, N - 1, 24).astype(int)])).astype(np.int32)
    F = steps.force_eval(d, x, M, h)
    e = rel_err(F[rows], oracle.forces_rows(p, x, M, h, rows))
    report(f"pair-symmetric t3 ewald ng={ng} N={N}", e)
    assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-9
    dm, keepm = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T, precision=steps.PREC_MIXED)
    em = rel_err(steps.force_eval(dm, x, M, h), F)
    report(f"pair-symmetric t3 ewald ng={ng} N={N} mixed vs fp64", em)
    assert np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5


@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("shape", [(40, 33), (64, 8)])
def test_s1r2_lookup_edges(steps, oracle, order, shape):
    """Odd and even z grids, pairs on the axis, half a period apart, beyond the
    last rho node, and particles outside the box, which take the general lookup."""
    N, L, Rsim = 3001, 100.0, 20.0
    print(f"case pair-symmetric s1r2 edges order={order} shape={shape}", flush=True)
    x, M, h, _ = particles("s1r2", N, 9)
    x[:, :2] *= 0.3
    x = x[np.argsort(np.hypot(x[:, 0], x[:, 1]), kind="stable")]
    x[100:160, :2] = x[100, :2]
    x[130:160, 2] = (x[100:130, 2] + L / 2 + 1e-9 * (np.arange(30) - 15)) % L
    nrho, nz = shape
    rho = np.arange(nrho)[:, None] * (2.25 * Rsim / (nrho - 1))
    z = (np.arange(nz)[None, :] + 0.5) * (L / nz) - 0.5 * L
    T = np.stack([1e-6 * rho * np.exp(-(z / L) ** 2), 1e-6 * z * np.exp(-rho / L)], axis=-1)
    T = np.ascontiguousarray(T.reshape(-1))
    kw = dict(is_periodic=2, L=L, Rsim=Rsim, s1r2_lookup=1, interp_order=order, s1r2_table=T, s1r2_shape=shape)
    for label, y in (("in the box", x), ("outside", x + np.where(np.arange(N)[:, None] % 7 == 0, [0.0, 0.0, 1.75 * L], 0.0))):
        d, keep = steps.make_desc(steps.TOPO_S1R2, **kw)
        F = steps.force_eval(d, y, M, h)
        rows = np.unique(np.concatenate([np.arange(95, 165), np.linspace(0, N - 1, 60).astype(int)])).astype(np.int32)
        e = rel_err(F[rows], oracle.forces_rows(oracle.params(2, **kw), y, M, h, rows))
        report(f"pair-symmetric s1r2 edges order={order} {shape} {label}", e)
        # pairs exactly half a period apart may take either image: the median only
        assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and np.percentile(e, 80) <= 1e-9
        dm, keepm = steps.make_desc(steps.TOPO_S1R2, precision=steps.PREC_MIXED, **kw)
        em = rel_err(steps.force_eval(dm, y, M, h), F)
        report(f"pair-symmetric s1r2 edges order={order} {shape} {label} mixed vs fp64", em)
        assert np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5


@pytest.mark.parametrize("N", [MIN_N, MIN_N + 63, 10 * 1024 - 1, 15 * 1024, 33000])
@pytest.mark.parametrize("mode", ["r3", "t3", "s1r2"])
def test_equal_masses_against_oracle(steps, oracle, mode, N):
    """Particles of one mass, whose products leave the pairs: whole and ragged
    last blocks and tiles, close and coincident pairs; resident and one-shot
    calls, and the masses changed in between."""
    print(f"case pair-symmetric equal masses {mode} N={N}", flush=True)
    x, M, h, L = particles(mode, N, N)
    (d, keep), p = descriptor(steps, oracle, mode, L)
    rows = np.unique(np.concatenate([np.arange(0, 40), np.arange(N - 70, N),
                                     np.linspace(0, N - 1, 40).astype(int)])).astype(np.int32)
    sim = steps.Sim(d, N)
    for label, m in (("equal", np.full(N, 0.37)), ("mixed", M), ("equal again", np.full(N, 1.6))):
        F = steps.force_eval(d, x, m, h)
        e = rel_err(F[rows], oracle.forces_rows(p, x, m, h, rows))
        report(f"pair-symmetric equal masses {mode} N={N} {label}", e)
        assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-10
        sim.set_state(x, m, h)
        sim.forces()
        assert np.array_equal(sim.get_forces(), F)
        (dm, keepm), _ = descriptor(steps, oracle, mode, L)
        dm.precision = steps.PREC_MIXED
        em = rel_err(steps.force_eval(dm, x, m, h), F)
        report(f"pair-symmetric equal masses {mode} N={N} {label} mixed vs fp64", em)
        assert np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5 and em.max() <= 1e-3
