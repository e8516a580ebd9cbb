"""The conservation sums where their partition can go wrong -- fewer cells than workgroups, rows
shorter than a workgroup's width, chunks that start mid-row, one cell more than whole chunks -- in
both precisions and geometries, against exactly rounded sums (math.fsum) of the same terms.

Tolerance: the terms are formed with up to 8 roundings each and summed with compensation: 16 x 2^-53
of the sum of their magnitudes (all terms are positive)."""
import math

import numpy as np
import pytest

from asteriy_2d_amd import grid as G
from asteriy_2d_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geometry", [G.PLANAR, G.AXISYMMETRIC])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("N,M", [(2, 2), (2, 700), (5, 51), (16, 16), (1023, 3), (1024, 2),
                                 (1025, 257), (700, 2), (333, 401)])
def test_sums(dev, geometry, dtype, N, M):
    import torch
    from asteriy_2d_amd import solver
    g = G.Grid.from_extent(N, M, -1.0, 1.0, 1.0, gamma=5.0 / 3.0, krit=0.3, geometry=geometry,
                           bc=(G.BC_OUTFLOW,) * 4)
    s, u = problems.random_state(g, seed=N * M)
    s, u = (a.astype(dtype) for a in (s, u))
    print(f"sums {N}x{M} {dtype} geometry={geometry}", flush=True)
    got = solver.conservation_sums(g, torch.from_numpy(s).to(dev), torch.from_numpy(u).to(dev))
    s, u = s.astype(np.float64), u.astype(np.float64)
    w = np.full(M, g.dx * g.dy) * (g.y(np.arange(M)) if geometry == G.AXISYMMETRIC else 1.0)
    E = s[..., 1] / (g.gamma - 1.0) + 0.5 * s[..., 0] * (u ** 2).sum(-1)
    want = [math.fsum((s[..., 0] * w[:, None]).ravel()), math.fsum((E * w[:, None]).ravel())]
    for a, b in zip(got.tolist(), want):
        assert abs(a - b) <= 16 * 2.0 ** -53 * b
