"""Mixed-precision R3 forces do not depend on the units: lengths times 2^a and
masses times 2^b scale every FP32 quantity by a power of two, so the forces are
those of the unscaled particles times 2^(b - 2a), also where r^-3 itself is
outside the FP32 range (2^40 AU is 5 Mpc): to the bit, but for the order of two
products in the pair-symmetric kernel where masses differ."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("a,b", [(40, 60), (42, 44), (-44, -50)])
@pytest.mark.parametrize("masses", ["equal", "different"])
@pytest.mark.parametrize("N", [3000, 14335, 14337, 66001])
def test_forces_scale_with_the_units(steps, N, masses, a, b):
    print(f"case mixed units {masses} N={N} lengths 2^{a} masses 2^{b}", flush=True)
    rng = np.random.default_rng(N)
    x = rng.normal(size=(N, 3)) * 30.0
    x[1:200:2] = x[0:199:2] + rng.normal(size=(100, 3)) * 0.02          # pairs inside the softening length
    M = rng.uniform(0.5, 2.0, N) if masses == "different" else np.full(N, 1.375)
    h = np.full(N, 0.03)
    d, keep = steps.make_desc(steps.TOPO_R3, precision=steps.PREC_MIXED)
    F = steps.force_eval(d, x, M, h)
    d64, keep64 = steps.make_desc(steps.TOPO_R3)
    F64 = steps.force_eval(d64, x, M, h)
    e = np.linalg.norm(F - F64, axis=1) / np.linalg.norm(F64, axis=1)
    assert np.median(e) <= 2e-6 and np.percentile(e, 99) <= 1e-5          # the mixed path's bar
    G = np.ldexp(steps.force_eval(d, np.ldexp(x, a), np.ldexp(M, b), np.ldexp(h, a)), 2 * a - b)
    if masses == "equal" or N < 14336:
        assert np.array_equal(G, F)
    e = np.linalg.norm(G - F64, axis=1) / np.linalg.norm(F64, axis=1)
    assert np.median(e) <= 2e-6 and np.percentile(e, 99) <= 1e-5
