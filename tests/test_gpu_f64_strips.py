"""The FP64 step's strips where they can go wrong, against the CPU oracle to the 1e-12 bar: grids
of one partial band, whole bands and one column more; both ghost columns of a side in one band;
every ghost rule on every side; strips that do not divide the rows; frozen cells in some waves
only; grids whose default strip height the rule changes."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

from cases import PARITY_REL, step_mismatch

pytestmark = pytest.mark.gpu

STATE = [[1.2, 0.9, 0.8, 0.1], [0.7, 1.4, -0.6, -0.2], [1.1, 0.8, 0.2, 0.5], [0.9, 1.2, -0.1, -0.4]]
KINDS = [G.BC_OUTFLOW, G.BC_REFLECT, G.BC_DIRICHLET, G.BC_OUTFLOW_CLAMPED, G.BC_DIRICHLET_PULSED]


def _grid(N, M, kinds, **kw):
    return G.Grid.from_extent(N, M, -1.0, 1.0, 1.0, gamma=5.0 / 3.0, krit=0.3, bc=kinds,
                              bc_state=STATE, bc_vclamp=(-0.2, 0.3, 0.1, -0.1),
                              bc_pulse=(0.3, 2.0, 0.6, 1.0), **kw)


def _check(dev, ora, g, s, u, method, T_do=2e-3, TT=0.4, rows=None):
    import torch
    from asteriy_2d_amd import solver
    from asteriy_2d_amd.sim import Simulation
    print(f"step_f64 {g.N}x{g.M} bc={tuple(g.bc)} method={method} rows={rows}", flush=True)
    rs, ru, rT = ora.step(g, s, u, 1e7, T_do, method, TT=TT)
    if rows is None:
        t = lambda a: torch.tensor(a, dtype=torch.float64, device=dev)
        S, U = t(s), t(u)
        S2, U2 = torch.empty_like(S), torch.empty_like(U)
        T = t([1e7])
        solver.Kernel_TVD(g, S, U, S2, U2, T, t([T_do]), t([TT]), method)
        s2, u2, T = S2.cpu().numpy(), U2.cpu().numpy(), float(T.item())
    else:
        with Simulation(g, method, "f64", s, u) as sim:
            sim.set_time(1e7, T_do, TT, 0)
            sim.set_tile_rows(rows)
            sim.run(1, graph=False)
            s2, u2 = sim.state()
            T = sim.time()["T_do"]  # the step's minimum, taken by the time advance
    bad, worst = step_mismatch(s2, u2, rs, ru, g.gamma)
    assert bad == 0, (bad, worst)
    assert abs(T - rT) <= PARITY_REL * rT


@pytest.mark.parametrize("N,M", [(2, 2), (3, 5), (59, 4), (60, 3), (61, 7), (62, 9), (120, 2), (121, 13)])
def test_sizes_and_rows(dev, ora, N, M):
    g = _grid(N, M, (G.BC_DIRICHLET, G.BC_OUTFLOW_CLAMPED, G.BC_REFLECT, G.BC_OUTFLOW),
              geometry=G.AXISYMMETRIC)
    s, u = problems.random_state(g, seed=N + M)
    for rows in (None, 1, 2, 3, 5, 70):
        _check(dev, ora, g, s, u, G.HLLC, rows=rows)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("side", range(4))
def test_ghost_rules(dev, ora, kind, side):
    kinds = [G.BC_REFLECT, G.BC_OUTFLOW, G.BC_OUTFLOW, G.BC_REFLECT]
    kinds[side] = kind
    g = _grid(64, 11, tuple(kinds))
    s, u = problems.random_state(g, seed=side)
    for method in (G.HLL, G.HLLC_A):
        _check(dev, ora, g, s, u, method)
    _check(dev, ora, g.replace(ho_lo=-0.5, ho_hi=0.5), s, u, G.HLLC, rows=4)


@pytest.mark.parametrize("N,M,rows", [(200, 40, 3), (130, 64, None), (130, 70, 70)])
def test_frozen_cells_in_some_waves(dev, ora, N, M, rows):
    g = _grid(N, M, (G.BC_OUTFLOW, G.BC_DIRICHLET, G.BC_REFLECT, G.BC_OUTFLOW),
              geometry=G.AXISYMMETRIC, frozen_x0=0.1, frozen_ax=0.2, frozen_ay=0.3)
    s, u = problems.random_state(g, seed=3)
    _check(dev, ora, g, s, u, G.HLLC, rows=rows)


# the default height's rule: one row (few waves), 3 and 5 rows (one and two waves a SIMD), 7 (three),
# and taller strips in rounds; more than 64 rows a strip re-reads the radii
@pytest.mark.parametrize("N,M,rows", [(256, 128, None), (512, 256, None), (1024, 512, None),
                                      (1500, 751, None), (2048, 1023, None), (300, 400, 150)])
def test_default_heights(dev, ora, N, M, rows):
    p = problems.wind(N, M)
    _check(dev, ora, p.grid, p.s, p.u, G.HLLC, T_do=1e-2, rows=rows)


def test_time_left_below_the_steps_minimum(dev):
    """A T set below what the first step would find is what that step leaves (Kernel_TVD lowers
    the *T it is given), for that step alone."""
    from asteriy_2d_amd.sim import Simulation
    p = problems.wind(64, 32)
    with Simulation(p.grid, G.HLLC, "f64", p.s, p.u) as sim:
        sim.run(2)
        free = sim.time()["T_do"]
        for graph in (False, True):
            sim.set_state(p.s, p.u)
            sim.set_time(0.25 * free, 1e-9, 0.0, 0)
            sim.run(1, graph=graph)
            assert sim.time()["T_do"] == 0.25 * free
            sim.set_state(p.s, p.u)
            sim.set_time(0.25 * free, 1e-9, 0.0, 0)
            sim.run(20, graph=graph)
            t = sim.time()
            assert t["T"] == 1e7 and t["T_do"] > 0.5 * free and t["i"] == 20
