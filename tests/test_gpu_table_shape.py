"""One buffer read as S1R2 tables of two shapes with the same number of nodes:
each call takes the shape it names."""
import numpy as np
import pytest

from conftest import rel_err, report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [0, 2, 4])
def test_shape_of_the_same_buffer(steps, oracle, order):
    print(f"case table shape order {order}", flush=True)
    N, L, Rsim = 1500, 100.0, 20.0
    rng = np.random.default_rng(3)
    x = rng.uniform(0.0, L, (N, 3))
    x[:, :2] = (x[:, :2] - 50.0) * 0.5
    M, h = rng.uniform(0.5, 2.0, N), np.full(N, 0.03)
    T = np.ascontiguousarray(1e-6 * rng.normal(size=33 * 9 * 2))
    rows = np.arange(0, N, 15).astype(np.int32)
    # the layout of the first shape is the larger one
    for shape in ((33, 9), (9, 33), (33, 9)):
        kw = dict(is_periodic=2, L=L, Rsim=Rsim, s1r2_lookup=1, interp_order=order, s1r2_table=T, s1r2_shape=shape)
        d, keep = steps.make_desc(steps.TOPO_S1R2, **kw)
        F = steps.force_eval(d, x, M, h)
        e = rel_err(F[rows], oracle.forces_rows(oracle.params(2, **kw), x, M, h, rows))
        report(f"table shape {shape} order {order}", e)
        # the FP64 bars of the table tests
        assert np.median(e) <= 1e-12 and np.percentile(e, 90) <= 1e-9
