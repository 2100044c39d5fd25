"""The coordinate MLP's row tiles at the edges of their ranges: one row, row
counts beside a tile and beside the switches between tile heights, every
width in steps of 64 up to the widest tile and beyond it (the layer-by-layer
products), one and 64 outputs; and one training step against the gradient.
Tolerances as for the network's other numerics: activations, weights and
gradients round to BF16 (2^-9 relative) at the same points in both, so what
differs is the rounding of values whose FP32 sums differ in the last bits."""
import os
import sys

import numpy as np
import pytest

from product_util import ROOT, glhip

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import mlp_ref as R  # noqa: E402

pytestmark = pytest.mark.gpu
G = glhip()


def _rel(a, b):
    return float(np.linalg.norm(np.asarray(a, np.float64) - b) / max(np.linalg.norm(b), 1e-300))


@pytest.mark.parametrize("F,W,D,n_out,n", [(32, 64, 1, 1, 1), (64, 192, 2, 18, 33), (128, 256, 3, 64, 65),
                                           (64, 128, 7, 33, 1000), (32, 320, 2, 18, 100), (160, 256, 1, 18, 70),
                                           (64, 256, 2, 18, 16383), (64, 192, 1, 18, 57344), (64, 256, 2, 18, 57345)])
def test_tiles_match_reference(F, W, D, n_out, n):
    print("mlp tile", F, W, D, n_out, n, flush=True)
    net = G.MLP(n_freq=F, sigma=1.0, width=W, depth=D, n_out=n_out, seed=5)
    try:
        p, B = net.params()
        rng = np.random.default_rng(n)
        X = rng.uniform(-1, 1, (n, 6)).astype(np.float32)
        Y = rng.standard_normal((n, n_out)).astype(np.float32)
        assert _rel(net.predict(X), R.predict(p, B, X, F, W, D, n_out)) <= 5e-3
        L, g = net.loss_grad(X, Y)
        Lr, gr = R.loss_grad(p, B, X, Y, F, W, D, n_out)
        assert L == pytest.approx(Lr, rel=2e-3)
        K, N, offs, _ = R.layout(F, W, D, n_out)
        for (a, b), m in zip(offs, N):
            assert _rel(g[a:b], gr[a:b]) <= 2e-2 and _rel(g[b:b + m], gr[b:b + m]) <= 2e-2
    finally:
        net.close()


@pytest.mark.parametrize("W,batch", [(64, 64), (256, 192), (192, 20480), (256, 57344)])
def test_first_training_step_is_adams(W, batch):
    """One data point: the batch's gradient is that point's, and Adam's first
    step is lr g / (|g| + 1e-8) (FP32: a few units of 2^-24 of the step and of
    the parameter; 1e-3 of lr covers both)."""
    print("mlp step", W, batch, flush=True)
    net = G.MLP(n_freq=32, sigma=1.0, width=W, depth=2, n_out=18, seed=1)
    try:
        rng = np.random.default_rng(W)
        X = rng.uniform(-1, 1, (1, 6)).astype(np.float32)
        Y = rng.standard_normal((1, 18)).astype(np.float32)
        p0, _ = net.params()
        L0, g = net.loss_grad(np.repeat(X, batch, 0), np.repeat(Y, batch, 0))
        net.set_data(X, Y)
        L = net.train(1, batch=batch, lr=1e-3, seed=2, loss_every=1)
        p1, _ = net.params()
        assert L[0] == pytest.approx(L0, rel=1e-5)
        # gradients near Adam's epsilon would turn their own rounding into a step
        big = np.abs(g) > 1e-5
        assert big.mean() > 0.3
        step = 1e-3 * g[big].astype(np.float64) / (np.abs(g[big]) + 1e-8)
        assert np.max(np.abs((p0[big].astype(np.float64) - p1[big]) - step)) <= 1e-6
        # the next step runs on the updated BF16 weights
        assert net.loss_grad(X, Y)[0] < L0
    finally:
        net.close()
