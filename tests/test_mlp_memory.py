"""The device memory of a gradient, with the library's host code on
hip_host.cpp's runtime (no GPU, no kernels)."""
import pytest

import hip_host


@pytest.mark.parametrize("width,depth", [(64, 1), (256, 2), (256, 5), (192, 7), (320, 5)])
def test_gradient_needs_no_more_than_layer_by_layer(width, depth):
    # What the layer-by-layer form of the network takes a row: the points and
    # targets, the BF16 activations and FP32 pre-activations of every layer,
    # the outputs and their gradient (64 columns), the gradients of two layers; and
    # a partial sum of the loss for four rows.
    # A gradient that fits the card so is not refused by the row tiles.
    hip_host.run("""
width, depth, n = %d, %d, 1 << 16
net = G.MLP(n_freq=32, sigma=1.0, width=width, depth=depth, n_out=18, seed=1)
X, Y = np.zeros((n, 6), np.float32), np.zeros((n, 18), np.float32)
net.loss_grad(X[:64], Y[:64])  # the splits' partials and whatever else the rows do not change
n0 = H.hh_used()
row = 4 * (6 + 18) + 2 * (64 + depth * width) + 4 * depth * width + 64 * (4 + 2) + 2 * 2 * width
H.hh_limit(n0 + (n - 64) * row + n + 4096)
net.loss_grad(X, Y)
assert H.hh_bad() == 0
""" % (width, depth))
