"""The FP32 exact flux at the ends of its range, against the FP64 one: NaN words, sides without
pressure, units that put products of words near the smallest FP32 numbers."""
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


@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.3])
def test_two_shocks_into_a_side_without_pressure(dev, gamma):
    """p = 0 on one side, the speeds closing: the reference's Newton is NaN there (its start is p =
    0) and its comparisons sample the side with pressure, at the floor of the wave speed."""
    n = 20000
    F = _faces(n, 2)
    F[5] = 0.0
    sr = np.sqrt(F[1] / (0.5 * F[4] * (gamma + 1.0)))  # f_I(p_II)
    F[6] = F[2] - sr * np.random.default_rng(3).uniform(1.1, 5.0, n)
    F[:, ::2] = F[:, ::2][[4, 5, 6, 7, 0, 1, 2, 3]]    # the other way round
    F[[2, 6], ::2] *= -1.0
    X, a, b = _pair(F, dev, gamma=gamma)
    K = np.where(X[1] > 0.0, X[:4], X[4:])             # the side with pressure
    m = K[0] * K[2]
    side = np.stack([m, (gamma / (gamma - 1.0) * K[1] + 0.5 * K[0] * (K[2] ** 2 + K[3] ** 2)) * K[2],
                     m * K[2] + K[1], m * K[3]])
    assert np.allclose(b[:4], side, rtol=1e-12, atol=0.0)
    assert np.allclose(a[:4], side, rtol=2e-6, atol=0.0)  # products of FP32 words
    assert np.allclose(a[4], b[4], rtol=1e-6)


def small_units(n, seed):
    """Faces in units that leave products of a density and a pressure at the end of the FP32
    range: r and p over eight decades around 1e-18."""
    rng = np.random.default_rng(seed)
    F = np.empty((8, n))
    for k in (0, 1, 4, 5):
        F[k] = 10.0 ** rng.uniform(-22.0, -14.0, n)
    c = np.sqrt(np.maximum(F[1] / F[0], F[5] / F[4]))
    for k in (2, 3, 6, 7):
        F[k] = rng.uniform(-5.0, 5.0, n) * c
    return F


def fraction_within(X, a, b, gamma, tol=1e-2):
    """The fraction of faces whose five values lie within tol of the FP64 ones (or of the lighter
    side's flux scale, a thousandth of it)."""
    v = np.abs(X[[2, 3, 6, 7]]).max(axis=0) + np.sqrt(gamma * np.maximum(X[1] / X[0], X[5] / X[4]))
    r = 1e-3 * np.minimum(X[0], X[4])
    S = np.maximum(np.abs(b), np.stack([r * v, r * v ** 3, r * v ** 2, r * v ** 2, 0.0 * v]))
    with np.errstate(invalid="ignore", over="ignore"):
        return float((np.abs(a - b) <= tol * S).all(axis=0).mean())


# the fractions with the p* solves of sums of products (rK ((g+1) p + (g-1) pK)): 0.854, 0.844,
# 0.840; with those of ratios of pressures, 0.863, 0.854, 0.849 (the rest are faces whose mass
# fluxes a_K leave the range themselves)
@pytest.mark.parametrize("gamma,least", [(5.0 / 3.0, 0.8621), (1.4, 0.8532), (1.3, 0.8489)])
def test_small_units(dev, gamma, least):
    X, a, b = _pair(small_units(400000, 4), dev, gamma=gamma)
    assert fraction_within(X, a, b, gamma) >= least
