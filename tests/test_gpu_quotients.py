"""The division and square root of the FP64 solvers on the device, read off the operators' dt =
krit*rad/max|wave speed|: bit for bit the IEEE quotient and root where flux64.hpp says so, and
infinities where a quotient overflows (v_div_fixup makes one of the NaN that its residual gives)."""
import numpy as np
import pytest

from asteriy_2d_amd import grid as G

pytestmark = pytest.mark.gpu

N = 1 << 20


def _dt(dev, method, r, p, u, rad, gamma):
    """dt of faces with equal sides at speed u (normal) and state r, p."""
    import torch

    from asteriy_2d_amd import solver
    z = np.zeros_like(u)
    F = torch.from_numpy(np.stack([r, p, u, z, r, p, u, z])).to(dev)
    return solver.flux_batch(method, F, 1.0, 0.0, rad, gamma=gamma, krit=1.0)[4].cpu().numpy()


def _wide(rng, n, span):
    return np.ldexp(rng.uniform(1.0, 2.0, n), rng.integers(-span, span, n))


def test_quotients_are_ieee(dev):
    """A sound speed below the rounding of u leaves the speed u itself (side velocities of every
    binade; c = 2^-60 u): dt = rad/u."""
    rng = np.random.default_rng(0)
    u = _wide(rng, N, 200) * rng.choice([-1.0, 1.0], N)
    p = np.ldexp(0.6 * u * u, -120)
    for rad in (1.0, 3.0e-91, 0.7e107):
        got = _dt(dev, G.HLLC, np.ones(N), p, u, rad, 5.0 / 3.0)
        assert np.array_equal(got, rad / np.abs(u))


@pytest.mark.parametrize("method", [G.HLL, G.HLLC, G.HLLC_A])
def test_roots_are_ieee(dev, method):
    """At rest the speed is c = sqrt(gamma p / r); gamma p is exact for gamma = 2.  HLL caps its
    dt at 1e7."""
    rng = np.random.default_rng(1)
    p, r = _wide(rng, N, 100), _wide(rng, N, 100)
    got = _dt(dev, method, r, p, np.zeros(N), 1.0, 2.0)
    want = 1.0 / np.sqrt(2.0 * p / r)
    assert np.array_equal(got, np.minimum(want, 1e7) if method == G.HLL else want)


@pytest.mark.parametrize("method", [G.HLLC, G.HLLC_A, G.EXACT])
def test_overflow_is_infinite(dev, method):
    u = np.full(1000, 1e-10)
    got = _dt(dev, method, np.ones(1000), np.full(1000, 1e-30), u, 1e302, 5.0 / 3.0)
    assert np.isposinf(got).all()
    assert np.isposinf(_dt(dev, method, np.ones(70000), np.full(70000, 1e-30),
                           np.full(70000, 1e-10), 1e302, 5.0 / 3.0)).all()


def test_mhd_overflow_is_infinite(dev):
    import torch

    from asteriy_2d_amd import solver
    n = 1000
    F = torch.zeros((18, n), dtype=torch.float64, device=dev)
    for k in (0, 9):
        F[k], F[k + 1], F[k + 2], F[k + 6] = 1.0, 1.0, 1e-30, 1e-16
    for method in (G.HLLC_MHD, G.HLLD):
        out = solver.flux_mhd_batch(method, F, 1.0, 0.0, 0.0, 1e302, krit=1.0)
        assert torch.isposinf(out[9]).all()


def test_smallest_denominators(dev):
    """Down to 2^-1024 (not included) a denominator may be subnormal; at and below it the quotient
    is infinite, as for a denominator of zero."""
    rng = np.random.default_rng(2)
    u = np.ldexp(rng.uniform(1.0, 2.0, N), rng.integers(-1023, -1019, N))
    got = _dt(dev, G.HLLC, np.ones(N), np.zeros(N), u, 0.037, 5.0 / 3.0)
    assert np.array_equal(got, 0.037 / u)
    got = _dt(dev, G.HLLC, np.ones(N), np.zeros(N), np.full(N, 2.0 ** -1024), 2.0 ** -30, 5.0 / 3.0)
    assert np.isposinf(got).all()
