"""The training kernels at the edges of their tiles, against the numpy network: batches of less
than, exactly and one more than the 16 samples of a wave's block, the 128 of a workgroup's and the
32768 of the grid's first pass, with and without a mask, the masked and clamped rows holding
features that must not count; and the MFMA operands an Adam step leaves.

Tolerance: FP32 sums of n rounded products of size up to S lie within a few n^(1/2) 2^-24 S of
their value; with the mean taken, every entry is bounded by 1e-5 of the gradient's largest (as a
hardware tanh of relative error 1e-6 allows), the loss by 1e-5 of itself."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NPARAM = 2369


def _case(n, seed):
    from asteriy_2d_amd import learned
    rng = np.random.default_rng(seed)
    return (learned.glorot_init(seed), rng.normal(size=(n, 6)).astype(np.float32),
            rng.normal(size=n).astype(np.float32))


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 127, 128, 129, 32768, 32769, 40001])
def test_gradient_at_tile_edges(dev, n, masked):
    import torch
    from asteriy_2d_amd.learned import LearnedGuess
    from oracle import mlp_ref as R
    p, X, t = _case(n, n)
    m = None
    if masked:
        m = (np.random.default_rng(n + 1).random(n) < 0.6).astype(np.uint8)
        t[m == 0] = 1e6  # a masked row's target must not count
    print(f"loss_grad n={n} masked={masked}", flush=True)
    model = LearnedGuess(p)
    a = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(dev)
    loss, grad = model.loss_grad(a(X.T), a(t), None if m is None else a(m))
    if m is not None and m.sum() == 0:
        assert loss.item() == 0.0 and not grad.any()
        return
    lref, gref = R.loss_grad(p.astype(np.float64), X.astype(np.float64), t.astype(np.float64), m)
    g = grad.cpu().numpy()
    assert abs(loss.item() - lref) <= 1e-5 * abs(lref)
    assert np.abs(g - gref).max() <= 1e-5 * np.abs(gref).max()


def test_adam_leaves_the_operands_of_its_masters(dev):
    """After an Adam step on a block whose operands were never built, the BF16 forward equals the
    one of a fresh block with the same masters."""
    import torch
    from asteriy_2d_amd.learned import LearnedGuess
    p, X, t = _case(512, 5)
    model = LearnedGuess(p)
    model.buffer[4 * NPARAM:] = 0x5A  # stale operand bytes
    g = torch.from_numpy(np.random.default_rng(2).normal(size=NPARAM).astype(np.float32)).to(dev)
    model.adam(g, torch.zeros(2 * NPARAM, device=dev), 1, 1e-2)
    other = LearnedGuess(model.params())
    assert not np.array_equal(model.params(), p)
    f = torch.from_numpy(np.ascontiguousarray(X.T)).to(dev)
    assert torch.equal(model.forward(f), other.forward(f))
