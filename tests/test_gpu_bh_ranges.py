"""Octree walks split into ranges of the item list: particle counts on both
sides of the rule's steps, fewer items than ranges, and the least scratch (one
range), against the oracle's octree and each other."""
import ctypes as C

import numpy as np
import pytest

from conftest import rel_err, report
from steps_amd import _abi
from steps_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [2, 31, 1000, 32769, 699051, 1048577])
def test_ranges_against_oracle(steps, oracle, N):
    print(f"case octree ranges N={N}", flush=True)
    w = wl.r3_compactified(N=N, seed=N)
    kw = dict(cosmology=1, comoving=1, mass_in_unit_sphere=w.mass_in_unit_sphere)
    d, keep = steps.make_desc(steps.TOPO_R3, bh_theta=0.5, bh_particle_radius=w.particle_radius, **kw)
    F = steps.force_eval(d, w.x, w.M, w.soft)
    assert np.all(np.isfinite(F))
    for lo in sorted({0, N // 2, max(0, N - 300)}):
        hi = min(N, lo + 300) - 1
        Fo = oracle.forces_bh_ex(oracle.params(0, **kw), 0.5, w.particle_radius, w.x, w.M, w.soft, id_min=lo, id_max=hi)
        e = rel_err(F[lo:hi + 1], Fo)
        report(f"octree ranges N={N} rows {lo}..{hi}", e)
        # FP64 bars of every path: median 1e-12 (summation order), max 1e-10
        assert np.median(e) <= 1e-12 and e.max() <= 1e-10
    assert np.array_equal(steps.force_eval(d, w.x, w.M, w.soft), F)


def test_one_range_and_many_agree(steps):
    """steps_force_eval_noalloc (256 MiB) has to do with one range where
    steps_force_eval takes several: the same interactions."""
    N = 690000
    print(f"case octree ranges, least scratch N={N}", flush=True)
    w = wl.r3_compactified(N=N, seed=5)
    d, keep = steps.make_desc(steps.TOPO_R3, bh_theta=0.5, bh_particle_radius=w.particle_radius)
    F = steps.force_eval(d, w.x, w.M, w.soft)
    lib = steps.load_library()
    G = np.zeros(3 * N)
    x, M, h = (np.ascontiguousarray(a, dtype=np.float64) for a in (w.x.reshape(-1), w.M, w.soft))
    rc = lib.steps_force_eval_noalloc(C.byref(d), N, _abi._ptr(x), _abi._ptr(M), _abi._ptr(h), _abi._ptr(G), 0, N - 1)
    assert rc == 0, lib.steps_last_error()
    e = rel_err(G.reshape(-1, 3), F)
    report(f"octree one range vs ranges N={N}", e)
    assert np.median(e) <= 1e-12 and e.max() <= 1e-10
