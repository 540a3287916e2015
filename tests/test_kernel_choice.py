"""Which kernel an evaluation takes, on both sides of every threshold.
Launches are counted by name on a host-memory runtime."""
import pytest

import fake_hip

DESC = """
L = 100.0
def table(odd):
    g = (np.arange(20) - 9.5) * (L / 20)
    T = np.stack(np.meshgrid(g, g, g, indexing="ij"), axis=-1) * 1e-6
    if not odd:
        T[3, 4, 5, 2] = 1.0
    return np.ascontiguousarray(T.reshape(-1))
def cylinder(odd):
    nr, nz = 24, 16
    rho = np.arange(nr)[:, None] * (2.25 * 80.0 / (nr - 1))
    z = (np.arange(nz)[None, :] + 0.5) * (L / nz) - 0.5 * L
    T = np.stack([1e-6 * rho + 0 * z, 1e-6 * z + 0 * rho], axis=-1)
    if not odd:
        T[5, 3, 1] = 1.0
    return dict(s1r2_lookup=1, s1r2_table=np.ascontiguousarray(T.reshape(-1)), s1r2_shape=(nr, nz))
KINDS = {
    "r3": lambda p: steps.make_desc(steps.TOPO_R3, precision=p),
    "t3": lambda p: steps.make_desc(steps.TOPO_T3, is_periodic=1, L=L, precision=p),
    "s1r2": lambda p: steps.make_desc(steps.TOPO_S1R2, is_periodic=1, L=L, Rsim=80.0, precision=p),
    "ewald": lambda p: steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=table(True), precision=p),
    "ewald-bent": lambda p: steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=table(False), precision=p),
    "cic": lambda p: steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, interp_order=2, precision=p, **cylinder(True)),
    "tsc": lambda p: steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, interp_order=4, precision=p, **cylinder(True)),
    "ngp": lambda p: steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, interp_order=0, precision=p, **cylinder(True)),
    "cic-bent": lambda p: steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=80.0, interp_order=2, precision=p, **cylinder(False)),
}
for kind, precision, N, rows in CASES:
    d, keep = KINDS[kind](precision)
    fake.fake_reset_launches()
    steps.force_eval(d, *cloud(N, L), id_min=0, id_max=rows - 1)
    one = launches("pair_kernel")
    sym = {k: launches(k) for k in ("sym_kernel", "sym_mixed_kernel", "sym_t3_kernel", "sym_s1r2_kernel")}
    names = [k for k, n in sym.items() if n] + (["pair_kernel"] if one else [])
    print(kind, precision, N, rows, *names)
"""

# (topology, precision, N, rows): the kernel
EXPECT = {
    ("r3", 0, 8191, 8191): "pair_kernel", ("r3", 0, 8192, 8192): "sym_kernel",
    ("r3", 0, 9000, 6000): "sym_kernel", ("r3", 0, 9000, 5999): "pair_kernel",
    ("r3", 1, 14335, 14335): "pair_kernel", ("r3", 1, 14336, 14336): "sym_mixed_kernel",
    ("t3", 0, 8191, 8191): "pair_kernel", ("t3", 0, 8192, 8192): "sym_kernel",
    ("t3", 1, 14335, 14335): "pair_kernel", ("t3", 1, 14336, 14336): "sym_mixed_kernel",
    ("s1r2", 0, 8191, 8191): "pair_kernel", ("s1r2", 0, 8192, 8192): "sym_kernel",
    ("s1r2", 1, 20000, 20000): "pair_kernel",          # mixed: the one-sided kernel at every N
    ("ewald", 0, 127, 127): "pair_kernel", ("ewald", 0, 128, 128): "sym_t3_kernel",
    ("ewald", 1, 127, 127): "pair_kernel", ("ewald", 1, 128, 128): "sym_t3_kernel",
    ("ewald-bent", 0, 3000, 3000): "pair_kernel", ("ewald-bent", 1, 3000, 3000): "pair_kernel",
    ("cic", 0, 1023, 1023): "pair_kernel", ("cic", 0, 1024, 1024): "sym_s1r2_kernel",
    ("cic", 1, 1023, 1023): "pair_kernel", ("cic", 1, 1024, 1024): "sym_s1r2_kernel",
    ("tsc", 0, 1024, 1024): "sym_s1r2_kernel", ("tsc", 1, 1024, 1024): "sym_s1r2_kernel",
    ("ngp", 0, 9000, 9000): "pair_kernel", ("cic-bent", 0, 9000, 9000): "pair_kernel",
}


def test_kernels(tmp_path):
    got = {}
    for line in fake_hip.run(tmp_path, f"CASES = {list(EXPECT)!r}\n" + DESC):
        kind, precision, N, rows, *names = line.split()
        got[kind, int(precision), int(N), int(rows)] = "+".join(names)
    assert got == EXPECT


@pytest.mark.gpu
@pytest.mark.parametrize("N", [14335, 14336, 14337])
@pytest.mark.parametrize("mode", ["r3", "t3"])
def test_mixed_on_both_sides_of_its_threshold(steps, mode, N):
    import numpy as np

    from conftest import rel_err, report

    print(f"case mixed threshold {mode} N={N}", flush=True)
    rng = np.random.default_rng(N)
    x = rng.uniform(0.0, 100.0, (N, 3))
    x[1:200:2] = x[0:199:2] + rng.normal(size=(100, 3)) * 0.02
    if mode == "t3":
        x %= 100.0
    M, h = rng.uniform(0.5, 2.0, N), np.full(N, 0.03)
    make = {"r3": lambda p: steps.make_desc(steps.TOPO_R3, precision=p),
            "t3": lambda p: steps.make_desc(steps.TOPO_T3, is_periodic=1, L=100.0, precision=p)}[mode]
    F, G = (steps.force_eval(make(p)[0], x, M, h) for p in (steps.PREC_FP64, steps.PREC_MIXED))
    e = rel_err(G, F)
    report(f"mixed threshold {mode} N={N}", e)
    # the bars of the mixed path: median 2e-6, p99 1e-5 of the pair sum, and the image every pair takes
    assert np.median(e) <= 2e-6 and np.percentile(e, 99) <= 1e-5 and e.max() <= 1e-3
    assert not np.array_equal(G, F) and np.array_equal(steps.force_eval(make(1)[0], x, M, h), G)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n_side", [16, 25])
def test_t3_window_kernel_against_the_global_one(steps, n_side, precision):
    """A table that is not odd: the full evaluation takes the one-sided kernel
    with the table window, all rows but 37 the one that reads the table from
    memory; the same sums."""
    import numpy as np

    from steps_amd import workloads as wl

    print(f"case t3 window n_side={n_side} precision {precision}", flush=True)
    w = wl.t3_lattice(n_side=n_side, seed=1001)
    T = steps.t3_table(2, w.L).reshape(63, 63, 63, 3).copy()
    T[:, :, 40:, 2] *= 1.25
    d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=w.L, t3_table=T.reshape(-1), precision=precision)
    F = steps.force_eval(d, w.x, w.M, w.soft)
    G = steps.force_eval(d, w.x, w.M, w.soft, id_min=37, id_max=w.N - 1)
    assert np.array_equal(G, F[37:])
