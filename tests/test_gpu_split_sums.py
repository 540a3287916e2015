"""The sums over source splits of the one-sided kernels: split counts around
the number the reduction loads at once, ragged last workgroups of rows."""
import numpy as np
import pytest

from conftest import rel_err, report
from steps_amd import workloads as wl

pytestmark = pytest.mark.gpu


# one tile of 64 sources a split below N = 4096, two from there
@pytest.mark.parametrize("N", [2, 63, 64, 65, 448, 512, 513, 1024, 1089, 4095, 4096, 8191])
def test_split_counts_against_oracle(steps, oracle, N):
    print(f"case split sums N={N}", flush=True)
    w = wl.r3_compactified(N=N, seed=N)
    kw = dict(cosmology=1, comoving=1, mass_in_unit_sphere=w.mass_in_unit_sphere)
    d, keep = steps.make_desc(steps.TOPO_R3, **kw)
    F = steps.force_eval(d, w.x, w.M, w.soft)
    rows = np.unique(np.concatenate([np.arange(min(N, 70)), np.arange(max(0, N - 70), N)])).astype(np.int32)
    e = rel_err(F[rows], oracle.forces_rows(oracle.params(0, **kw), w.x, w.M, w.soft, rows))
    report(f"split sums N={N}", e)
    # FP64 bars of every path: median 1e-12 (summation order), max 1e-10
    assert np.all(np.isfinite(F)) and np.median(e) <= 1e-12 and e.max() <= 1e-10
    part = steps.force_eval(d, w.x, w.M, w.soft, id_min=N // 3, id_max=N // 2)
    e = rel_err(part, F[N // 3:N // 2 + 1])
    assert np.median(e) <= 1e-12 and e.max() <= 1e-10
