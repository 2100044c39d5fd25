"""The weight gradients' large tiles (a launch of 512 workgroups or more) on
distinct samples: a sum that pairs one sample's activations with another's
output gradient, or takes a step of samples twice, is wrong there.
Tolerances as for the row tiles: both sides round to BF16 (2^-9 relative) at
the same points, so what differs is the rounding of values whose FP32 sums
differ in the last bits; mispaired samples are wrong by the gradient itself."""
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


# 1032 steps of 32 samples in 32 splits, the last of 9 steps instead of 33, and
# 20 tiles: 640 workgroups; 1088 steps in 32 whole splits of 34 and 21 tiles of
# which some are partly filled; below the switch: 640 steps in 24 splits, 480
@pytest.mark.parametrize("F,W,D,n_out,n", [(64, 256, 5, 18, 33001), (128, 192, 5, 64, 34816), (64, 256, 5, 18, 20433)])
def test_gradient_of_distinct_rows(F, W, D, n_out, n):
    print("mlp large tiles", F, W, D, n_out, n, flush=True)
    net = G.MLP(n_freq=F, sigma=1.0, width=W, depth=D, n_out=n_out, seed=3)
    try:
        p, B = net.params()
        rng = np.random.default_rng(n)
        X = rng.uniform(-1, 1, (n, 6)).astype(np.float32)
        Y = rng.standard_normal((n, n_out)).astype(np.float32)
        L, g = net.loss_grad(X, Y)
        Lr, gr = R.loss_grad(p, B, X, Y, F, W, D, n_out)
        assert L == pytest.approx(Lr, rel=2e-3)
        K, N, offs, _ = R.layout(F, W, D, n_out)
        for (a, b), m in zip(offs, N):
            assert _rel(g[a:b], gr[a:b]) <= 2e-2 and _rel(g[b:b + m], gr[b:b + m]) <= 2e-2
    finally:
        net.close()


def _mix64(z):
    z = z + np.uint64(0x9E3779B97F4A7C15)
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


@pytest.mark.parametrize("W,D,batch", [(256, 2, 57344), (256, 5, 65536), (192, 3, 20480)])
def test_first_training_step_on_distinct_points(W, D, batch):
    """The rows a step draws are hash(seed, step, row) mod n; the first Adam
    step on them is lr g / (|g| + 1e-8) of their gradient g."""
    print("mlp step on distinct points", W, D, batch, flush=True)
    F, n, seed, lr = 64, 5000, 2, 1e-3
    net = G.MLP(n_freq=F, sigma=1.0, width=W, depth=D, n_out=18, seed=1)
    try:
        rng = np.random.default_rng(W + D)
        X = rng.uniform(-1, 1, (n, 6)).astype(np.float32)
        Y = np.tanh(X @ rng.standard_normal((6, 18))).astype(np.float32)
        with np.errstate(over="ignore"):
            h = _mix64(np.uint64(seed) ^ _mix64(np.uint64(1 << 32) | np.arange(batch, dtype=np.uint64)))
        rows = (h % np.uint64(n)).astype(np.int64)
        assert len(np.unique(rows)) > 0.9 * n
        p0, B = net.params()
        Lr, gr = R.loss_grad(p0, B, X[rows], Y[rows], F, W, D, 18)
        net.set_data(X, Y)
        L = net.train(1, batch=batch, lr=lr, seed=seed, loss_every=1)
        p1, _ = net.params()
        assert L[0] == pytest.approx(Lr, rel=2e-3)
        d = p0.astype(np.float64) - p1
        K, N, offs, _ = R.layout(F, W, D, 18)
        for (a, b), m in zip(offs, N):
            gl, dl = gr[a:b + m], d[a:b + m]
            # an entry above a tenth of the largest is not moved by a tenth of
            # itself by roundings of 2e-2 of the layer's norm; the step then by
            # 0.1 g 1e-8 / (0.9 g + 1e-8)^2 of lr (FP32, with the parameter's
            # own rounding: 1e-4 of lr)
            ga = np.abs(gl)
            big = ga > 0.1 * ga.max()
            assert big.sum() >= 10
            step = lr * gl[big] / (ga[big] + 1e-8)
            tol = lr * (1e-9 * ga[big] / (0.9 * ga[big] + 1e-8) ** 2 + 1e-4)
            assert np.all(np.abs(dl[big] - step) <= tol)
            # and elsewhere the sign is the gradient's for nearly all
            assert np.mean(np.sign(dl) == np.sign(gl)) >= 0.9
    finally:
        net.close()
