"""The order in which the network's gradient is summed (k_mlp_grad, k_mlp_adam):
a tile's samples four by four and the fours in pairs, the tiles of a block and
the blocks one after another. Training passes the rounding of these sums on
from step to step, so the order is part of what a training call returns.

The gradient is scaled by 2 / batch. Between batches of powers of two that is
an exact factor, BF16 copies included, so the gradient of a batch is the sum of
its parts' gradients to the last bit, in the stated order.
"""
import numpy as np
import pytest

import pydem

pytestmark = pytest.mark.gpu

BIASES = np.r_[1152:1216, 5312:5376, 5568:5571]  # b1, b2, b3 behind W1, W2, W3


def _solver():
    rng = np.random.default_rng(3)
    s = pydem.SqSolver()
    s.net_init(seed=5)
    p = s.net_params()
    s.set_net_params(p + rng.normal(0, 0.05, p.shape).astype(np.float32))
    return s, rng


def _serial(parts):
    total = np.zeros_like(parts[0])
    for p in parts:
        total = total + p
    return total


@pytest.mark.parametrize("blocks", [2, 16, 32, 64, 128, 256, 512])
def test_blocks_are_added_one_after_another(blocks):
    n = 64 * blocks
    print(f"[gpu] gradient of {n} samples against its blocks of 64", flush=True)
    s, rng = _solver()
    X = rng.normal(0, 1, (n, 18)).astype(np.float32)
    T = rng.normal(0, 0.5, (n, 3)).astype(np.float32)
    whole, loss = s.net_gradient(X, T)
    part = [s.net_gradient(X[k:k + 64], T[k:k + 64]) for k in range(0, n, 64)]
    s.close()
    scale = np.float32(1.0 / blocks)
    assert np.array_equal(whole, _serial([g * scale for g, _ in part]))
    assert np.float32(loss) == _serial([np.float32(v) for _, v in part]) * scale


def test_samples_of_a_tile():
    print("[gpu] bias gradients of 16 samples against the single ones", flush=True)
    s, rng = _solver()
    X = rng.normal(0, 1, (16, 18)).astype(np.float32)
    T = rng.normal(0, 0.5, (16, 3)).astype(np.float32)
    whole, _ = s.net_gradient(X, T)
    one = [s.net_gradient(X[k:k + 1], T[k:k + 1])[0][BIASES] * np.float32(1 / 16) for k in range(16)]
    s.close()
    four = [_serial(one[k:k + 4]) for k in range(0, 16, 4)]
    assert np.array_equal(whole[BIASES], (four[0] + four[1]) + (four[2] + four[3]))
