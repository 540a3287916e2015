"""Mixed precision: a pair whose FP32 r^2 lies at the limit below which pairs
are done again in FP64 has its force once, whichever way r^2 rounds.  The kernels that
form the displacement in FP64, where a pair's own force is good to 1e-5."""
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

f32 = np.float32


def fma32(a, b, c):
    return f32(float(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c))))


def r2_orders(d):
    """FP32 r^2 by the orders x y z, x z y, z y x ... of its fused sum."""
    x, y, z = (f32(v) for v in d)
    return [fma32(a, a, fma32(b, b, f32(c * c))) for a, b, c in
            ((x, y, z), (z, x, y), (z, y, x), (x, z, y), (y, x, z), (y, z, x))]


def limits(rng, box):
    """(position, displacement, softening length) with the limit ((2 h (1 +
    1e-5))^2 in FP32) between the least and the largest r^2."""
    while True:
        p = rng.uniform(0.3, 0.7, 3) * box
        q = p + rng.uniform(0.02, 0.08, 3)
        v = r2_orders(q - p)
        if min(v) == max(v):
            continue
        b = f32(np.sqrt(float(max(v))))
        for _ in range(3):
            h = float(b) / (2.0 * (1.0 + 1e-5))
            if f32((h + h) * (1.0 + 1e-5)) == b and min(v) < f32(b * b) <= max(v):
                yield p, q, h
                break
            b = np.nextafter(b, f32(1.0))


def cases(steps):
    L, Rsim = 100.0, 80.0
    s1 = dict(is_periodic=2, L=L, Rsim=Rsim, s1r2_lookup=1)
    T, shape = steps.s1r2_table(2, L, Rsim)
    E = steps.t3_table(2, L)
    return {
        "t3-ewald": (700, lambda p: steps.make_desc(steps.TOPO_T3, is_periodic=2, L=L, t3_table=E, precision=p)),
        "s1r2-cic": (1100, lambda p: steps.make_desc(steps.TOPO_S1R2, interp_order=2, s1r2_table=T, s1r2_shape=shape,
                                                     precision=p, **s1)),
        "s1r2-tsc": (1100, lambda p: steps.make_desc(steps.TOPO_S1R2, interp_order=4, s1r2_table=T, s1r2_shape=shape,
                                                     precision=p, **s1)),
    }


@pytest.mark.parametrize("path", ["t3-ewald", "s1r2-cic", "s1r2-tsc"])
def test_one_force_at_the_limit(steps, path):
    L = 100.0
    N, make = cases(steps)[path]
    rng = np.random.default_rng(7)
    for k, (p, q, h) in zip(range(24), limits(rng, L)):
        print(f"case close limit {path} {k}", flush=True)
        x = rng.uniform(0.0, L, (N, 3))
        near = np.linalg.norm(x - p, axis=1) < 1.0          # the pair's own force is the largest by far
        x[near] = rng.uniform(0.0, 0.2 * L, (int(near.sum()), 3))
        i, j = (int(v) for v in rng.choice(N, 2, replace=False))
        x[i], x[j] = p, q
        M, soft = np.full(N, 1.0) + 0.1 * rng.random(N), np.full(N, h)
        (d, keep), (dm, keepm) = make(steps.PREC_FP64), make(steps.PREC_MIXED)
        F, G = steps.force_eval(d, x, M, soft), steps.force_eval(dm, x, M, soft)
        for row in (i, j):
            e = np.linalg.norm(G[row] - F[row]) / np.linalg.norm(F[row])
            assert e <= 1e-5, (path, k, row, e)             # the mixed path's bar
