"""The batch's runs where its time protocol can go wrong: runs of 1, 19, 20, 21 and 45 steps in a
row (captured chunks, remainders, starts from either plane), graph and direct launches, instances
of very different sizes (fewer rows than a strip, one partial band), both kinds of solver -- bit for
bit the single-grid runtime, with equal times; and a T left below the first step's minimum."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu

SIZES = [(61, 2), (130, 6), (300, 150), (64, 33), (500, 120)]


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("method", [G.HLLC, G.EXACT])
def test_runs_equal_single_grids(dev, method, graph):
    from asteriy_2d_amd.batch import Batch
    from asteriy_2d_amd.sim import Simulation
    inst = [problems.wind(N, M) for N, M in SIZES]
    print(f"batch method={method} graph={graph}", flush=True)
    with Batch([p.grid for p in inst], method, [(p.s, p.u) for p in inst]) as b:
        for n in (1, 19, 20, 21, 45):
            b.run(n, graph=graph)
        got = [(b.state(k), b.time(k)) for k in range(len(inst))]
    for p, ((s, u), t) in zip(inst, got):
        with Simulation(p.grid, method, "f32", p.s, p.u) as sim:
            sim.run(106, graph=False)
            a, c = sim.state()
            assert np.array_equal(s, a) and np.array_equal(u, c)
            assert t == sim.time()


def test_time_left_below_the_steps_minimum(dev):
    from asteriy_2d_amd.batch import Batch
    p = problems.wind(64, 32)
    with Batch([p.grid] * 2, G.HLLC, [(p.s, p.u)] * 2) as b:
        b.run(1)
        free = b.time(0)["T_do"]
        for k in range(2):
            b.set_state(k, p.s, p.u)
            b.set_time(k, 0.25 * free if k else 1e7, 1e-9, 0.0, 0)
        b.run(1)
        assert b.time(0)["T_do"] == free and b.time(1)["T_do"] == 0.25 * free
        b.run(24)
        assert b.time(1)["T"] == 1e7 and b.time(1)["T_do"] > 0.5 * free and b.time(1)["i"] == 25
