"""Rows within an ulp of a cube's opening limit: the walks of all item ranges
decide alike, so the cube's force counts once, whichever way r^2 rounds.

One particle has all the mass, so every cube that holds it has its position as
centre of mass to the bit, and the root, which holds the first items of most
ranges, is taken where side^2 / theta^2 < r^2.  The opening angle is chosen so
that the limit is the smaller of the two values that r^2 has by two orders of
its fused sum."""
from fractions import Fraction

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N, R0, TINY = 4001, 64.0, 2.0 ** -80


def fma(a, b, c):
    return float(Fraction(a) * Fraction(b) + Fraction(c))


def cloud(seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-30.0, 30.0, (N, 3))
    x[0] = (R0, 0.0, 0.0)                               # the largest radius: the root's side
    heavy = N // 2
    M = np.full(N, TINY)
    M[heavy] = 1.0
    return x, M, np.full(N, 1e-6), heavy


def borderline(x, heavy, side):
    """(row, theta) with the limit at the smaller of the row's two r^2."""
    for i in range(1, N):
        dx, dy, dz = (float(x[heavy, c] - x[i, c]) for c in range(3))
        a, b = fma(dz, dz, fma(dx, dx, dy * dy)), fma(dz, dz, fma(dy, dy, dx * dx))
        if i == heavy or a == b:
            continue
        theta = side / np.sqrt(min(a, b))
        for k in range(-40, 41):
            t = theta + k * np.spacing(theta)
            if (side * side) * (1.0 / (t * t)) == min(a, b):
                yield i, t, a < b
                break


@pytest.mark.parametrize("first_smaller", [True, False])
def test_one_force_at_the_limit(steps, first_smaller):
    x, M, h, heavy = cloud(3)
    done = 0
    for i, theta, order in borderline(x, heavy, 2.00002 * R0):
        if order != first_smaller:
            continue
        print(f"case octree limit row {i} theta {theta!r}", flush=True)
        d, keep = steps.make_desc(steps.TOPO_R3, bh_theta=float(theta), bh_particle_radius=1e-12)
        F = steps.force_eval(d, x, M, h)
        dr = x[heavy] - x[i]
        expect = dr / np.linalg.norm(dr) ** 3
        # r^-3 within 2.1e-14, the rest of the mass is 2^-68
        assert np.linalg.norm(F[i] - expect) <= 1e-12 * np.linalg.norm(expect), (F[i], expect)
        done += 1
        if done == 6:
            break
    assert done == 6
