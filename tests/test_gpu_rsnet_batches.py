"""Learned-radius training kernels at the batch sizes where their work split
changes: part of a 16-sample group, of a 64-sample block, and more blocks
than partial rows (16384 samples); epochs whose last minibatch is ragged."""
import numpy as np
import pytest

from nbody6ppgpu_amd import rsnet
from oracle import mlp_ref as M
from test_gpu_rsnet import data, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 16384, 16385, 16449])
def test_grad_at_block_edges(n):
    """Against the checker.  One BF16 rounding that falls the other way (the
    kernels' exp is hardware exp2) moves a hidden unit by 2^-8 of itself, so
    a gradient over a few samples by about 1e-2 at most; over hundreds such
    flips average out (test_gpu_rsnet.py's 3e-3)."""
    rng = np.random.default_rng(60 + n)
    X, t = data(rng, n)
    if n == 1:
        X, t = np.repeat(X, 2, 0), np.repeat(t, 2)
    p, norm = setup(rng, X, t)
    X, t = X[:n], t[:n]
    L, g = rsnet.grad(X, t)
    Lr, gr = M.loss_and_grad(p, norm, X, t, emulate=True)
    tol = 3e-3 if n > 100 else 2e-2
    assert abs(L - Lr) <= tol * Lr
    for a, b in ((M.OW1, M.OB1), (M.OB1, M.OW2), (M.OW2, M.OB2),
                 (M.OB2, M.OW3), (M.OW3, M.OB3), (M.OB3, M.NP)):
        blk = np.linalg.norm(g[a:b] - gr[a:b]) / max(np.linalg.norm(gr[a:b]), 1e-12)
        assert blk < tol, (a, b, blk)


@pytest.mark.parametrize("n,batch", [(1000, 300), (1000, 1000), (130, 1), (5000, 4999)])
def test_epoch_loss_of_ragged_minibatches(n, batch):
    """With a step of zero length the epoch's loss is the loss over all
    samples (FP32 sums per row: 1e-5 relative), and the parameters stay."""
    rng = np.random.default_rng(90 + n)
    X, t = data(rng, n)
    p, _ = setup(rng, X, t)
    L, _ = rsnet.grad(X, t)
    Le = rsnet.train(X, t, epochs=2, batch=batch, lr=0.0, seed=2)
    assert abs(Le - L) <= 1e-5 * L
    assert np.array_equal(rsnet.get_params(), p)
