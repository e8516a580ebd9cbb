"""The FP32 tilings chosen by the grid's size against 8-row strips, bit for bit (the sizes where
the rules change: strips of 4 rows, equal strips of 1 to 4 waves a SIMD, rounds; the exact
solver's 1 to 8 rows)."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M", [(64, 32), (512, 256), (768, 384), (1024, 512), (1500, 750),
                                 (600, 3000), (3000, 40)])
@pytest.mark.parametrize("method", [G.HLLC, G.EXACT])
def test_by_size_against_eight_rows(dev, N, M, method):
    from asteriy_2d_amd import native
    from asteriy_2d_amd.sim import Simulation
    assert native.load().ast_get_tile_rows() == 8  # every test before this one set it back
    p = problems.wind(N, M)
    got = []
    for tile in (None, 8):
        with Simulation(p.grid, method, "f32", p.s, p.u) as sim:
            if tile:
                sim.set_tile_rows(tile)
            sim.run(3)
            got.append((*sim.state(), sim.time()))
    a, b = got
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and a[2] == b[2]
