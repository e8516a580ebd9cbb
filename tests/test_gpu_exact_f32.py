"""The FP32 exact flux: its two kernels (faces in the batch's order, faces sorted
by wave pattern) against each other, and its p* solves over the gas constants
that take different code for the powers, against the FP64 solver."""
import numpy as np
import pytest

from asteriy_2d_amd import facegen
from asteriy_2d_amd import grid as G

pytestmark = pytest.mark.gpu


def _faces(n, seed, dev, **kw):
    import torch
    return torch.from_numpy(np.ascontiguousarray(facegen.faces(n, seed=seed, **kw))).to(dev).float()


def test_kernels_agree_bit_for_bit(dev):
    """Batches above 2^20 faces and counted ones are solved in sorted tiles,
    the others face by face: the same bits, whole and partial tiles alike."""
    import torch
    from asteriy_2d_amd import solver
    n = (1 << 20) + 700
    F = _faces(n, 31, dev)
    whole = solver.flux_batch(G.EXACT, F, 0.6, 0.8).cpu()
    for lo, hi in ((0, 1 << 20), (1 << 20, n), (n - 1, n), (12345, 12345 + 513)):
        part = solver.flux_batch(G.EXACT, F[:, lo:hi].contiguous(), 0.6, 0.8).cpu()
        assert torch.equal(part, whole[:, lo:hi]), (lo, hi)
    counted = solver.flux_batch(G.EXACT, F[:, :1500].contiguous(), 0.6, 0.8,
                                stats=solver.new_stats(dev)).cpu()
    assert torch.equal(counted, whole[:, :1500])


@pytest.mark.parametrize("counted", [False, True])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 2.0, 3.0, 1.25, 1.3, 1.1])
def test_gas_constants_against_f64(dev, gamma, counted):
    """n = 2 gamma/(gamma - 1): 5, 7 (products), 4, 3, 10 (loops), 8.67 and 22
    (the power function).  p = pII y^n, so an error of y counts n times: the
    bounds are those of the flux test at gamma 5/3, n/5 times (at least once)."""
    from asteriy_2d_amd import native, solver
    F = _faces(1 << 17, 32, dev)
    st = solver.new_stats(dev)
    o64 = solver.flux_batch(G.EXACT, F.double(), gamma=gamma).cpu().numpy()
    o32 = solver.flux_batch(G.EXACT, F, gamma=gamma, stats=st if counted else None)
    o32 = o32.double().cpu().numpy()
    rel = np.abs(o32[:4] - o64[:4]) / (np.abs(o64[:4]).max(axis=0) + 1e-30)
    k = max(1.0, 2.0 * gamma / (gamma - 1.0) / 5.0)
    for q, tol in ((0.5, 1e-7), (0.99, 1e-5), (0.999, 1e-4)):
        assert np.quantile(rel, q) < k * tol, (q, float(np.quantile(rel, q)))
    dt = np.abs(o32[4] - o64[4]) / o64[4]
    assert np.quantile(dt, 0.99) < k * 1e-4
    if counted:
        d = native.stats_from_tensor(st)
        assert d["capped"] == 0 and d["exact_faces"] == F.shape[1]
        assert min(d["newton_faces"], d["bisect_faces"], d["rarefaction_faces"]) > 100


def test_no_pattern_and_empty_sides(dev):
    """NaN words give NaN fluxes; a side at rest without pressure, and equal
    sides, give finite ones."""
    import torch
    from asteriy_2d_amd import solver
    one = [1.0, 1.0, 0.3, 0.1, 1.0, 1.0, 0.3, 0.1]
    F = torch.tensor([one] * 10, dtype=torch.float32, device=dev).t().contiguous()
    for k in range(8):
        F[k, k] = float("nan")
    F[1, 8] = 0.0
    o = solver.flux_batch(G.EXACT, F).cpu()
    assert bool(torch.isnan(o[:4, [0, 1, 2, 4, 5, 6]]).all())
    assert bool(torch.isfinite(o[:4, 8:]).all())
    m = 0.3  # rho u of equal sides
    assert abs(float(o[0, 9]) - m) < 1e-6
