"""The exact-solver steps of gases other than gamma = 5/3, which take kernels of their own (the
order 1/gm = 2 gamma/(gamma-1) read from the arguments: 7 and 4 as products, 8.67 by the power
function): FP64 against the oracle to the 1e-12 bar, FP32 against FP64 as the tests of gamma = 5/3
(3e-6 for states of order 1) and bit for bit over tilings, with the window, the counters, a
pulsed side and source planes."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

from cases import PARITY_REL, neutral_sources, step_mismatch

pytestmark = pytest.mark.gpu

STATE = [[1.2, 0.9, 0.8, 0.1], [0.7, 1.4, -0.6, -0.2], [1.1, 0.8, 0.2, 0.5], [0.9, 1.2, -0.1, -0.4]]
GASES = [1.4, 2.0, 1.3]
T_DO = 2e-3


def _grid(gamma, N=130, M=17, window=False, pulsed=False, geometry=G.AXISYMMETRIC):
    kw = dict(ho_lo=-0.5, ho_hi=0.4) if window else {}
    return G.Grid.from_extent(
        N, M, -1.0, 1.0, 1.0, gamma=gamma, krit=0.3, geometry=geometry,
        bc=(G.BC_DIRICHLET_PULSED if pulsed else G.BC_DIRICHLET, G.BC_OUTFLOW_CLAMPED, G.BC_REFLECT,
            G.BC_OUTFLOW), bc_state=STATE, bc_vclamp=(-0.2, 0.3, 0.1, -0.1),
        bc_pulse=(0.3, 2.0, 0.6, 1.0), **kw)


def _run(g, precision, s, u, tile=None, steps=1, counted=False, src=None):
    from asteriy_2d_amd.sim import Simulation
    print(f"exact {precision} gamma={g.gamma} {g.N}x{g.M} tile={tile} counted={counted} "
          f"src={src is not None}", flush=True)
    with Simulation(g, G.EXACT, precision, s, u) as sim:
        sim.set_time(1e7, T_DO, 0.4, 0)
        if tile is not None:
            sim.set_tile_rows(tile)
        if src is not None:
            sim.set_sources(*src, kmom=0.7, ken=0.02)
        sim.collect_stats(counted)
        sim.run(steps, graph=False)
        n = sim.stats()["exact_faces"]
        assert (n > 0) == counted
        return (*sim.state(), sim.time()["T_do"])


@pytest.mark.parametrize("window", [False, True])
@pytest.mark.parametrize("geometry", [G.AXISYMMETRIC, G.PLANAR])
@pytest.mark.parametrize("gamma", GASES)
def test_f64_against_the_oracle(dev, ora, gamma, geometry, window):
    for pulsed in (False, True):
        g = _grid(gamma, window=window, pulsed=pulsed, geometry=geometry)
        s, u = problems.random_state(g, seed=int(10 * gamma))
        rs, ru, rT = ora.step(g, s, u, 1e7, T_DO, G.EXACT, TT=0.4)
        for tile, counted in ((None, False), (1, False), (3, True), (17, False), (-2, True)):
            a, b, T = _run(g, "f64", s, u, tile, counted=counted)
            bad, worst = step_mismatch(a, b, rs, ru, g.gamma)
            assert bad == 0, (bad, worst)
            assert abs(T - rT) <= PARITY_REL * rT


@pytest.mark.parametrize("gamma", GASES)
def test_f64_counters_and_sources_change_no_bit(dev, gamma):
    g = _grid(gamma)
    s, u = problems.random_state(g, seed=6)
    src = neutral_sources(g.M, g.N)
    want = _run(g, "f64", s, u, 5, 3, False, src)
    for tile, counted in ((1, True), (-4, False), (17, True)):
        got = _run(g, "f64", s, u, tile, 3, counted, src)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert got[2] == want[2]


@pytest.mark.parametrize("kind", ["plain", "window", "pulsed", "sources"])
@pytest.mark.parametrize("gamma", GASES)
def test_f32_tilings_and_f64(dev, gamma, kind):
    g = _grid(gamma, window=kind == "window", pulsed=kind == "pulsed")
    s, u = problems.random_state(g, seed=4, smooth=True)
    src = neutral_sources(g.M, g.N) if kind == "sources" else None
    a, b, T = _run(g, "f32", s, u, 8, 1, False, src)
    c, d, T64 = _run(g, "f64", s, u, None, 1, False, src)
    assert np.abs(a - c).max() < 3e-6 and np.abs(b - d).max() < 3e-6
    assert abs(T - T64) < 1e-5 * T64
    want = _run(g, "f32", s, u, 8, 3, False, src)
    for tile, counted in ((1, False), (1, True), (3, False), (5, True), (70, False), (-3, False),
                          (-7, True), (None, False)):
        got = _run(g, "f32", s, u, tile, 3, counted, src)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert got[2] == want[2]


@pytest.mark.parametrize("gamma", GASES)
def test_batch_equals_single_grids(dev, gamma):
    from asteriy_2d_amd.batch import Batch
    from asteriy_2d_amd.sim import Simulation
    grids = [_grid(gamma, N, M) for N, M in ((61, 3), (130, 17), (300, 40))]
    states = [problems.random_state(g, seed=k, smooth=True) for k, g in enumerate(grids)]
    with Batch(grids, G.EXACT, states) as b:
        b.run(23)
        got = [(*b.state(k), b.time(k)) for k in range(3)]
    for g, (s, u), (a, c, t) in zip(grids, states, got):
        with Simulation(g, G.EXACT, "f32", s, u) as sim:
            sim.run(23)
            e, f = sim.state()
            assert np.array_equal(a, e) and np.array_equal(c, f) and t == sim.time()
