"""The FP32 step under every kind of tiling, bit for bit: one- to eight-row strips, strips taller
than the fast paths take, S strips a band, the tiling chosen by size; on grids of one partial band
to several, with fewer rows than a strip, every ghost rule, frozen cells and source planes.  And the
exact solver's one-row strips against the FP64 step: both solve the same Riemann problems, so a
step differs by FP32's rounding of states of order 1 (tests of the 8-row strips: 3e-6)."""
import subprocess
import sys

import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu

STATE = [[1.2, 0.9, 0.8, 0.1], [0.7, 1.4, -0.6, -0.2], [1.1, 0.8, 0.2, 0.5], [0.9, 1.2, -0.1, -0.4]]
BCS = [(G.BC_DIRICHLET, G.BC_OUTFLOW_CLAMPED, G.BC_REFLECT, G.BC_OUTFLOW),
       (G.BC_REFLECT, G.BC_DIRICHLET, G.BC_OUTFLOW_CLAMPED, G.BC_REFLECT),
       (G.BC_OUTFLOW_CLAMPED, G.BC_REFLECT, G.BC_DIRICHLET, G.BC_DIRICHLET)]
SIZES = [(62, 2), (121, 3), (64, 4), (130, 5), (59, 9), (200, 37), (61, 70)]


def _grid(N, M, bc, frozen=False):
    kw = dict(frozen_x0=0.1, frozen_ax=0.2, frozen_ay=0.3) if frozen else {}
    return G.Grid.from_extent(N, M, -1.0, 1.0, 1.0, gamma=5.0 / 3.0, krit=0.3,
                              geometry=G.AXISYMMETRIC, bc=bc, bc_state=STATE,
                              bc_vclamp=(-0.2, 0.3, 0.1, -0.1), **kw)


def _steps(g, method, precision, tile, s, u, src=None):
    from asteriy_2d_amd.sim import Simulation
    with Simulation(g, method, precision, s, u) as sim:
        sim.set_time(1e7, 2e-3, 0.0, 0)
        if src is not None:
            sim.set_sources(*src, ken=0.02)
        if tile is not None:
            sim.set_tile_rows(tile)
        sim.run(2, graph=False)
        a, b = sim.state()
        return a, b, sim.time()["TT"]


@pytest.mark.parametrize("method", [G.HLLC, G.EXACT])
@pytest.mark.parametrize("N,M", SIZES)
def test_tilings_bit_for_bit(dev, N, M, method):
    for k, bc in enumerate(BCS):
        g = _grid(N, M, bc, frozen=k == 0)
        s, u = problems.random_state(g, seed=k)
        src = None
        if k == 1:
            rng = np.random.default_rng(k)
            src = (rng.uniform(-0.1, 0.1, (M, N, 3)), rng.uniform(-0.1, 0.1, (M, N)))
        want = _steps(g, method, "f32", 8, s, u, src)
        for tile in (1, 2, 3, 4, 5, 64, 70, -1, -3, -7):
            if -tile > M:
                continue
            print(f"f32 {N}x{M} method={method} bc={bc} tile={tile}", flush=True)
            got = _steps(g, method, "f32", tile, s, u, src)
            assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
            assert got[2] == want[2]


@pytest.mark.parametrize("N,M", [(64, 4), (200, 37)])
def test_exact_one_row_strips_against_f64(dev, N, M):
    g = _grid(N, M, BCS[0])
    s, u = problems.random_state(g, seed=4, smooth=True)
    a, b, _ = _steps(g, G.EXACT, "f32", 1, s, u)
    c, d, _ = _steps(g, G.EXACT, "f64", 1, s, u)
    assert np.abs(a - c).max() < 3e-6 and np.abs(b - d).max() < 3e-6


SCRIPT = """
import numpy as np
from asteriy_2d_amd import grid as G, native, problems
from asteriy_2d_amd.sim import Simulation
L = native.load()
assert L.ast_get_tile_rows() == 8
sizes = [(64, 32), (512, 256), (768, 384), (1024, 512), (1500, 750), (600, 3000), (3000, 40)]
def run():
    out = []
    for N, M in sizes:
        for method in (G.HLLC, G.EXACT):
            p = problems.wind(N, M)
            with Simulation(p.grid, method, "f32", p.s, p.u) as sim:
                sim.run(3)
                out.append(sim.state())
    return out
a = run()
assert L.ast_set_tile_rows(8) == 0
b = run()
assert all(np.array_equal(x, y) for p, q in zip(a, b) for x, y in zip(p, q))
print("default tilings ok")
"""


def test_default_tilings(dev):
    """Before ast_set_tile_rows is called (a process of its own), the tiling chosen by size gives
    the bits of 8-row strips."""
    import os
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", SCRIPT], cwd=root, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0 and "default tilings ok" in r.stdout, r.stdout + r.stderr[-2000:]
