"""The FP32 exact flux on words its FP64 counterpart answers by the order of its comparisons:
NaN, and sides without pressure."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G

pytestmark = pytest.mark.gpu


def _pair(F, dev, **kw):
    """FP32 and FP64 fluxes of the same (FP32) faces."""
    import torch

    from asteriy_2d_amd import solver
    T = torch.from_numpy(F).to(dev).float()
    return (T.double().cpu().numpy(), solver.flux_batch(G.EXACT, T, **kw).double().cpu().numpy(),
            solver.flux_batch(G.EXACT, T.double(), **kw).cpu().numpy())


def _faces(n, seed):
    rng = np.random.default_rng(seed)
    F = np.empty((8, n))
    for k in (0, 1, 4, 5):
        F[k] = np.exp(rng.uniform(np.log(1e-3), np.log(1e3), n))
    c = np.sqrt(np.maximum(F[1] / F[0], F[5] / F[4]))
    for k in (2, 6):
        F[k] = rng.uniform(-5.0, 5.0, n) * c
    for k in (3, 7):
        F[k] = rng.uniform(-1.0, 1.0, n)
    return F


@pytest.mark.parametrize("n", [50000, (1 << 20) + 700])  # faces in order, sorted tiles
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.3])
def test_nan_is_not_lost(dev, n, gamma):
    """A face with one NaN word: NaN where the FP64 flux is."""
    F = _faces(n, 1)
    k = np.arange(n)
    F[k % 8, k] = np.nan
    _, a, b = _pair(F, dev, gamma=gamma)
    assert np.isnan(b[:4]).any(axis=0).sum() > n // 2
    assert np.isnan(a[:4])[np.isnan(b[:4])].all()
