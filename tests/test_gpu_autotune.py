"""What the autotuner reports is a tiling that another simulation can be given: the same steps, in
the tiling that was timed, in both precisions."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f32", "f64"])
@pytest.mark.parametrize("method", [G.HLLC, G.EXACT])
def test_reported_tiling_can_be_set(dev, precision, method):
    from asteriy_2d_amd import native
    from asteriy_2d_amd.sim import Simulation
    p = problems.wind(300, 64)

    def steps(tile):
        with Simulation(p.grid, method, precision, p.s, p.u) as sim:
            if tile is not None:
                sim.set_tile_rows(tile)
            sim.run(3)
            return (*sim.state(), sim.time())

    want = steps(None)
    with Simulation(p.grid, method, precision, p.s, p.u) as sim:
        for cand in ([-7], [5], [-64]):
            tile, us = sim.autotune(cand, reps=1)
            assert tile == cand[0] and 0 < us < 1e6
        tile, us = sim.autotune(reps=1)
        assert tile != 0 and us > 0
        for bad in (0, -65, 4097):
            with pytest.raises(native.AsteriyError):
                sim.set_tile_rows(bad)
    for t in (-7, 5, -64, tile):
        got = steps(t)
        assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert got[2] == want[2]
