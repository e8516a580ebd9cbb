"""A T left by set_time is what the first step of the next run lowers, and that step alone (the
*T of kernel.cu:3013-3017): the runtime against the protocol Kernel_TVD + funk_time from the same
T, bit for bit, however the run is cut into launches."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu

T_DO = 1e-9


def _protocol(p, method, dt, n, T0, dev):
    """n steps of Kernel_TVD + funk_time from T = T0: state, T_do, TT."""
    import torch

    from asteriy_2d_amd import solver
    S, U = (torch.from_numpy(a).to(dev).to(dt) for a in (p.s, p.u))
    S2, U2 = torch.empty_like(S), torch.empty_like(U)
    t = torch.tensor([T0, T_DO, 0.0], dtype=torch.float64, device=dev)
    for _ in range(n):
        solver.Kernel_TVD(p.grid, S, U, S2, U2, t[0:1], t[1:2], t[2:3], method)
        solver.funk_time(t[0:1], t[1:2], t[2:3])
        S, U, S2, U2 = S2, U2, S, U
    return S.double().cpu().numpy(), U.double().cpu().numpy(), t[1].item(), t[2].item()


@pytest.mark.parametrize("method", [G.HLLC, G.EXACT])
@pytest.mark.parametrize("precision", ["f32", "f64"])
def test_time_left_below_the_steps_minimum(dev, precision, method):
    import torch

    from asteriy_2d_amd.sim import Simulation
    dt = torch.float32 if precision == "f32" else torch.float64
    p = problems.wind(130, 70)
    free = _protocol(p, method, dt, 1, 1e7, dev)[2]
    with Simulation(p.grid, method, precision, p.s, p.u) as sim:
        for n in (1, 20, 40):
            s, u, t_do, tt = _protocol(p, method, dt, n, 0.25 * free, dev)
            for graph in (False, True):
                print(f"{precision} method={method} n={n} graph={graph}", flush=True)
                sim.set_state(p.s, p.u)
                sim.set_time(0.25 * free, T_DO, 0.0, 0)
                sim.run(n, graph=graph)
                a, b = sim.state()
                t = sim.time()
                assert t["T"] == 1e7 and t["T_do"] == t_do and t["TT"] == tt and t["i"] == n
                assert np.array_equal(a, s) and np.array_equal(b, u)


# positive IEEE doubles order like their bits, by which the step's atomic compares (on the
# protocol's *T as well), so these limit nothing
@pytest.mark.parametrize("T0", [-1.0, -0.0, float("nan")])
def test_negative_time_limits_nothing(dev, T0):
    from asteriy_2d_amd.batch import Batch
    from asteriy_2d_amd.sim import Simulation
    import torch
    p = problems.wind(62, 4)  # one workgroup
    for precision, dt in (("f32", torch.float32), ("f64", torch.float64)):
        want = _protocol(p, G.HLLC, dt, 1, T0, dev)[2]
        assert 0.0 < want < 1000.0
        with Simulation(p.grid, G.HLLC, precision, p.s, p.u) as sim:
            sim.set_time(T0, T_DO, 0.0, 0)
            sim.run(1)
            assert sim.time()["T_do"] == want, precision
        if precision == "f32":
            with Batch([p.grid], G.HLLC, [(p.s, p.u)]) as b:
                b.set_time(0, T0, T_DO, 0.0, 0)
                b.run(1)
                assert b.time(0)["T_do"] == want
