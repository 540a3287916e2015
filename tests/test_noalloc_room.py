"""steps_force_eval_noalloc takes every evaluation that fits its scratch with
the one-sided kernel and splits of 256 sources: finer splits and pair-symmetric
slots never make it refuse one.  On a host-memory runtime."""
import pytest

import fake_hip

RUN = """
import ctypes as C
from steps_amd import _abi
lib = steps.load_library()
def call(d, N, rows):
    x = np.random.default_rng(1).uniform(0.0, 100.0, 3 * N)
    M, h, F = np.ones(N), np.full(N, 0.01), np.zeros(3 * rows)
    return lib.steps_force_eval_noalloc(C.byref(d), N, _abi._ptr(x), _abi._ptr(M), _abi._ptr(h), _abi._ptr(F), 0, rows - 1)
"""


# a 205^3 table leaves 7 MiB beside itself and its device layout
@pytest.mark.parametrize("N,rows", [(8000, 8000), (9000, 9000), (10000, 7000), (12000, 4800)])
def test_fine_splits(tmp_path, N, rows):
    out = fake_hip.run(tmp_path, RUN + f"""
d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=100.0, t3_table=np.zeros(205 ** 3 * 3))
print(call(d, {N}, {rows}), call(d, 30000, 30000))
""")
    taken, refused = [int(v) for v in out[0].split()]
    assert taken == 0 and refused != 0


@pytest.mark.parametrize("N,share", [(468000, 0.7), (480000, 0.7), (488000, 0.67)])
def test_slots_of_one_cell(tmp_path, N, share):
    out = fake_hip.run(tmp_path, RUN + f"""
d, keep = steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=100.0, Rsim=80.0, s1r2_lookup=1, interp_order=2,
                          s1r2_table=np.zeros(2000 * 1500 * 2), s1r2_shape=(2000, 1500), precision=steps.PREC_MIXED)
print(call(d, {N}, {int(N * share)}), call(d, {N}, {N}))
""")
    taken, refused = [int(v) for v in out[0].split()]
    assert taken == 0 and refused != 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["fine splits", "slots of one cell"])
def test_forces_where_room_is_short(steps, case):
    import ctypes as C

    import numpy as np

    from conftest import rel_err, report
    from steps_amd import _abi

    print(f"case noalloc room: {case}", flush=True)
    if case == "fine splits":
        N, rows, bar = 8000, 8000, 1e-12
        d, keep = steps.make_desc(steps.TOPO_T3, is_periodic=2, L=100.0, t3_table=np.zeros(205 ** 3 * 3))
    else:
        N, rows, bar = 480000, 336000, 2e-6               # mixed: its median bar
        d, keep = steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=100.0, Rsim=80.0, s1r2_lookup=1, interp_order=2,
                                  s1r2_table=np.zeros(2000 * 1500 * 2), s1r2_shape=(2000, 1500),
                                  precision=steps.PREC_MIXED)
    rng = np.random.default_rng(1)
    x, M, h, F = rng.uniform(0.0, 100.0, 3 * N), rng.uniform(0.5, 2.0, N), np.full(N, 0.01), np.zeros(3 * rows)
    rc = steps.load_library().steps_force_eval_noalloc(C.byref(d), N, _abi._ptr(x), _abi._ptr(M), _abi._ptr(h),
                                                       _abi._ptr(F), 0, rows - 1)
    assert rc == 0
    G = steps.force_eval(d, x.reshape(-1, 3), M, h, id_min=0, id_max=rows - 1)
    e = rel_err(F, G)
    report(f"noalloc room {case}", e)
    assert np.all(np.isfinite(F)) and np.median(e) <= bar
