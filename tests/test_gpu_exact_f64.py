"""The FP64 exact flux's two kernels -- up to 2^16 faces in the batch's order, above
that (and for counted batches) sorted by wave pattern -- give the same bits."""
import numpy as np
import pytest

from asteriy_2d_amd import facegen
from asteriy_2d_amd import grid as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.3])
def test_kernels_agree_bit_for_bit(dev, gamma):
    import torch
    from asteriy_2d_amd import native, solver
    n = (1 << 16) + 700
    F = torch.from_numpy(np.ascontiguousarray(facegen.faces(n, seed=41))).to(dev)
    whole = solver.flux_batch(G.EXACT, F, 0.6, 0.8, gamma=gamma).cpu()
    for lo, hi in ((0, 1 << 16), (1 << 16, n), (n - 1, n), (1234, 1234 + 513)):
        part = solver.flux_batch(G.EXACT, F[:, lo:hi].contiguous(), 0.6, 0.8, gamma=gamma).cpu()
        assert torch.equal(part, whole[:, lo:hi]), (lo, hi)
    st = solver.new_stats(dev)
    counted = solver.flux_batch(G.EXACT, F[:, :1500].contiguous(), 0.6, 0.8, gamma=gamma, stats=st)
    assert torch.equal(counted.cpu(), whole[:, :1500])
    assert native.stats_from_tensor(st)["exact_faces"] == 1500
