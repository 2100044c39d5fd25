"""SiLU over the whole range of FP32, through the network: hidden biases z with
weights of 0, so that the layer's pre-activations are the biases, and an output
weight of 1e-37 or 1 on the neuron of each output.  Up to two roundings to BF16
(2^-9 each) of each output, of the activation and of the weight."""
import numpy as np
import pytest

from product_util import glhip

pytestmark = pytest.mark.gpu
G = glhip()

FMAX = float(np.finfo(np.float32).max)
Z = [8.4e37, FMAX / 4, 8.6e37, 1e38, 3.3e38, -8.6e37, -3.3e38, -FMAX, 33.0, 31.0, 17.0, 5.0, 1.0, 0.0, -1.0, -5.0,
     -87.0, -89.0]


@pytest.mark.parametrize("W,n", [(64, 5), (128, 20000), (256, 60000), (320, 70)])
def test_silu_of_every_size(W, n):
    print("silu", W, n, flush=True)
    F, N = 32, len(Z)
    net = G.MLP(n_freq=F, sigma=1.0, width=W, depth=1, n_out=N, seed=1)
    try:
        z = np.asarray(Z, np.float32)
        scale = np.where(np.abs(z) > 1e30, 1e-37, 1.0).astype(np.float32)
        b0 = np.zeros(W, np.float32)
        b0[:N] = z
        W1 = np.zeros((W, N), np.float32)
        W1[np.arange(N), np.arange(N)] = scale
        net.set_params(np.concatenate([np.zeros(2 * F * W, np.float32), b0, W1.reshape(-1), np.zeros(N, np.float32)]))
        X = np.random.default_rng(W).uniform(-1, 1, (n, 6)).astype(np.float32)
        z64 = z.astype(np.float64)
        ref = z64 / (1.0 + np.exp(-np.clip(z64, -700, 700))) * scale
        Y = net.predict(X)
        assert np.all(np.isfinite(Y))
        assert np.all(np.abs(Y - ref) <= 2.0 ** -7 * np.abs(ref) + 1e-36)
        # the gradient's sweep: the loss against the outputs, and finite
        L, g = net.loss_grad(X[:64], np.broadcast_to(ref.astype(np.float32), (64, N)))
        assert np.isfinite(L) and L <= np.mean((2.0 ** -7 * np.abs(ref)) ** 2) + 1e-30
        # d loss / d output bias is 2 (Y - T) / (n N) summed over the rows
        gb = g[-N:]
        assert np.all(np.isfinite(gb)) and np.all(np.abs(gb) <= 2 * 2.0 ** -7 * np.abs(ref) / N * 1.01 + 1e-30)
    finally:
        net.close()
