"""Resident simulations: row ranges of every size fit the scratch the
simulation was created with, and give the rows of the full evaluation; new
positions that are not finite are refused and change nothing, on both sides of
the size from which the device checks them."""
import numpy as np
import pytest

from conftest import rel_err
from steps_amd import _abi

pytestmark = pytest.mark.gpu


def cloud(N, seed, L):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, L, (N, 3))
    x[:, :2] -= L / 2
    return x, rng.uniform(0.5, 2.0, N), np.full(N, 0.03)


@pytest.mark.parametrize("N", [8300, 9000, 20000])
@pytest.mark.parametrize("order", [0, 2])
def test_row_ranges_fit(steps, order, N):
    """S1R2 NGP takes the one-sided kernel at every range, CIC changes over:
    a range may be split finer than the whole."""
    L, Rsim = 100.0, 150.0
    x, M, h = cloud(N, N, L)
    T, shape = steps.s1r2_table(2, L, Rsim)
    d, keep = steps.make_desc(steps.TOPO_S1R2, is_periodic=2, L=L, Rsim=Rsim, s1r2_lookup=1, interp_order=order,
                              s1r2_table=T, s1r2_shape=shape)
    sim = steps.Sim(d, N)
    sim.set_state(x, M, h)
    sim.forces()
    F = sim.get_forces()
    for rows in (1, 257, N // 3, 30 * 256, N - 300):
        rows = min(rows, N)
        print(f"case rows {rows} of {N} order {order}", flush=True)
        sim.forces(7 if rows < N - 7 else 0, rows - 1 + (7 if rows < N - 7 else 0))
        G = sim.get_forces()
        first = 7 if rows < N - 7 else 0
        # the same pairs in another order of summation: the FP64 bar
        assert np.median(rel_err(G[:rows], F[first:first + rows])) <= 1e-12


@pytest.mark.parametrize("N", [65535, 65536, 70001])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_positions_that_are_not_finite(steps, N, bad):
    print(f"case non-finite {bad} N={N}", flush=True)
    x, M, h = cloud(N, 3, 100.0)
    d, keep = steps.make_desc(steps.TOPO_R3)
    sim = steps.Sim(d, N)
    sim.set_state(x, M, h)
    for at in (0, 3 * N // 2, 3 * N - 1):
        y = x + 1.0
        y.reshape(-1)[at] = bad
        with pytest.raises(_abi.StepsError) as e:
            sim.set_positions(y)
        assert "non-finite" in str(e.value)
    assert np.array_equal(sim.get_state()[0], x)          # refused: the particles are as they were
    sim.set_positions(x + 1.0)                             # and the next ones are taken
    assert np.array_equal(sim.get_state()[0], x + 1.0)
