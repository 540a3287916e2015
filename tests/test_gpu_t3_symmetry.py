"""T3 tables by their symmetries: the pair-symmetric kernel looks |dz| up only
in a table that is mirrored in z at every node, the planes that a mirror maps
onto themselves included, and takes every other odd table as it stands."""
import numpy as np
import pytest

from conftest import rel_err, report

pytestmark = pytest.mark.gpu

L = 100.0


def grid(ng):
    g = (np.arange(ng) - (ng - 1) / 2) * (L / ng)
    return np.meshgrid(g, g, g, indexing="ij")


def mirrored(ng):
    X, Y, Z = grid(ng)
    f = 1e-6 * np.exp(-(X * X + Y * Y + Z * Z) / (0.1 * L * L))
    return np.stack([X * f, Y * f, Z * f], axis=-1)


def plane_x(ng):
    """Mirrored everywhere but on the plane x = 0 of an odd grid, where T_x is
    even in y and odd in z: still odd through the centre, still folded in x
    and y (the fold reads that plane as it is), not mirrored in z."""
    T = mirrored(ng)
    X, Y, Z = grid(ng)
    c = ng // 2
    T[c, :, :, 0] = 2e-5 * (Z * np.exp(-(Y * Y + Z * Z) / (0.1 * L * L)) / L)[c]
    return T


def plane_y(ng):
    T = mirrored(ng)
    X, Y, Z = grid(ng)
    c = ng // 2
    T[:, c, :, 1] = 2e-5 * (Z * np.exp(-(X * X + Z * Z) / (0.1 * L * L)) / L)[:, c]
    return T


def skew(ng):
    """T(-d) = -T(d) and no mirror in any axis."""
    X, Y, Z = grid(ng)
    f = 1e-6 * np.exp(-(X * X + Y * Y + Z * Z + 0.7 * X * Y + 0.5 * Y * Z - 0.4 * X * Z) / (0.1 * L * L))
    T = np.stack([(X + 0.3 * Z) * f, (Y - 0.4 * X) * f, (Z + 0.5 * Y) * f], axis=-1)
    half = T.reshape(-1, 3)[: (ng ** 3) // 2]
    flat = T.reshape(-1, 3)
    flat[ng ** 3 - 1 - np.arange(len(half))] = -half      # to the bit
    if ng % 2:
        flat[ng ** 3 // 2] = 0.0
    return T


def is_odd(T):
    flat = T.reshape(-1, 3)
    return bool(np.array_equal(flat[::-1], -flat))


def is_mirrored_z(T):
    M = T[:, :, ::-1] * np.array([1.0, 1.0, -1.0])
    return bool(np.array_equal(M, T))


def particles(N, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, L, (N, 3))
    x[1:100:2] = x[0:99:2] + rng.normal(size=(50, 3)) * 0.02
    x[200:260, 0] = 10.0 + 0.3 * (np.arange(60) % 5)       # close in x: stencils on the plane x = 0
    x[260:320, 1] = 20.0 + 0.3 * (np.arange(60) % 5)
    return x % L, rng.uniform(0.5, 2.0, N), np.full(N, 0.03)


# rows per workgroup 64, 128, 256 and 512 of the T3 Ewald kernel by particles
# per table column: N / ng^2 of 1 to 200
@pytest.mark.parametrize("table,ng,N", [
    (plane_x, 15, 700), (plane_x, 31, 3000), (plane_x, 63, 20011), (plane_x, 15, 30011),
    (plane_y, 15, 700), (plane_y, 31, 12007), (plane_y, 63, 40001),
    (skew, 3, 400), (skew, 8, 700), (skew, 15, 1087), (skew, 31, 3000), (skew, 62, 20011), (skew, 63, 20011),
    (skew, 31, 30011), (skew, 62, 66000), (skew, 63, 107001),
])
def test_odd_tables_against_oracle(steps, oracle, table, ng, N):
    print(f"case t3 symmetry {table.__name__} ng={ng} N={N}", flush=True)
    T4 = table(ng)
    assert is_odd(T4) and not is_mirrored_z(T4)
    T = np.ascontiguousarray(T4.reshape(-1))
    x, M, h = particles(N, N)
    rows = np.unique(np.concatenate([np.arange(200, 320, 7), np.linspace(0, N - 1, 24).astype(int)])).astype(np.int32)
    d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T)
    F = steps.force_eval(d, x, M, h)
    p = oracle.params(1, is_periodic=2, L=L, t3_table=T, interp_order=4)
    e = rel_err(F[rows], oracle.forces_rows(p, x, M, h, rows))
    report(f"t3 symmetry {table.__name__} ng={ng} N={N}", e)
    # the bars of every T3 Ewald test: FP64 median 1e-12, mixed p99 1e-5 of the pair sum
    assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-9
    assert np.array_equal(steps.force_eval(d, x, M, h), F)
    dm, keepm = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T, precision=steps.PREC_MIXED)
    Fm = steps.force_eval(dm, x, M, h)
    em = rel_err(Fm, F)
    report(f"t3 symmetry {table.__name__} ng={ng} N={N} mixed vs fp64", em)
    assert np.all(np.isfinite(Fm)) and np.median(em) <= 2e-6 and np.percentile(em, 99) <= 1e-5


def test_table_changed_between_calls(steps, oracle):
    """A mirrored table, one of its planes changed in place and changed back:
    each call takes the table as it is now, one-shot and resident."""
    ng, N = 15, 700
    print("case t3 symmetry, a table edited in place", flush=True)
    T = np.ascontiguousarray(mirrored(ng).reshape(-1))
    keep_T, other = T.copy(), plane_x(ng).reshape(-1)
    x, M, h = particles(N, 5)
    rows = np.arange(0, N, 11).astype(np.int32)
    d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T)
    first = steps.force_eval(d, x, M, h)
    for tab in (other, keep_T):
        T[:] = tab
        d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=T)
        F = steps.force_eval(d, x, M, h)
        e = rel_err(F[rows], oracle.forces_rows(oracle.params(1, is_periodic=2, L=L, t3_table=tab, interp_order=4),
                                                x, M, h, rows))
        assert np.median(e) <= 1e-12 and e.max() <= 1e-9
        sim = steps.Sim(d, N)
        sim.set_state(x, M, h)
        sim.forces()
        assert np.array_equal(sim.get_forces(), F)
    assert np.array_equal(F, first)
