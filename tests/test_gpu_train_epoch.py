"""The training kernels at the edges of their work split: rows per block with
and without a remainder, widths of several 32-pixel tiles, more tiles than
waves in the grid, and an epoch (losses read once at its end) against the same
batches one step at a time."""

import numpy as np
import pytest

from oracle import nn_oracle as O

pytestmark = pytest.mark.gpu


def _net(b, h, w):
    from exploringsycl_amd.nn import Net
    return Net(b, h, w)


def _data(seed, n, h, w):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, h, w, 3)).astype(np.float32),
            rng.standard_normal((n, h, w)).astype(np.float32))


# Rows of the batch: 15 (one per block), 279 (two per block, a short last
# one), 2048 (eight per block).
@pytest.mark.parametrize("b,h,w", [(3, 5, 96), (9, 31, 32), (64, 32, 32)])
def test_epoch_is_the_steps_one_by_one(b, h, w):
    x, t = _data(b, 2 * b + 1, h, w)
    order = np.random.default_rng(1).permutation(2 * b + 1).astype(np.int32)
    p = O.init_params(2)
    one, many = _net(b, h, w), _net(b, h, w)
    one.set_params(p)
    many.set_params(p)
    losses = [one.train_step(x[order[k:k + b]], t[order[k:k + b]], 1e-3)
              for k in (0, b)]
    many.load_dataset(x, t)
    mean = many.train_epoch(order, b, 1e-3)   # the short last batch is dropped
    assert mean == np.float32((float(losses[0]) + float(losses[1])) / 2)
    assert np.array_equal(one.get_params().view(np.int32), many.get_params().view(np.int32))


@pytest.mark.parametrize("b,h,w", [(3, 5, 96), (9, 31, 32)])
def test_gradients_match_the_oracle_at_uneven_splits(b, h, w):
    """The bound is test_gpu_nn.py's, for BF16 activations and deltas."""
    x, t = _data(7, b, h, w)
    p = O.init_params(3)
    net = _net(b, h, w)
    net.set_params(p)
    loss, g = net.loss_grad(x, t)
    loss_o, g_o = O.loss_grad(p, x, t, bf16_mode=True)
    assert abs(loss / loss_o - 1) < 2e-3
    k = 0
    for o, i in O.SHAPES:
        n = o * i * 9 + o
        assert np.linalg.norm(g[k:k + n] - g_o[k:k + n]) < 3e-2 * np.linalg.norm(g_o[k:k + n])
        k += n


def test_forward_of_more_tiles_than_waves_is_the_samples_one_by_one():
    """64 x 32 x 160: 10240 tiles on 8192 waves; each tile's MFMA sequence is
    that of a batch of one."""
    x, _ = _data(5, 64, 32, 160)
    net = _net(64, 32, 160)
    net.set_params(O.init_params(6))
    y = net.forward(x)
    for i in (0, 31, 51, 63):
        assert np.array_equal(y[i], net.forward(x[i:i + 1])[0])


def test_epoch_longer_than_the_set():
    """Samples drawn with repetition: ten batches from a set of five."""
    b, h, w = 4, 8, 32
    x, t = _data(11, 5, h, w)
    order = np.random.default_rng(2).integers(0, 5, 10 * b).astype(np.int32)
    p = O.init_params(4)
    one, many = _net(b, h, w), _net(b, h, w)
    one.set_params(p)
    many.set_params(p)
    losses = [one.train_step(x[order[k:k + b]], t[order[k:k + b]], 1e-3)
              for k in range(0, 10 * b, b)]
    many.load_dataset(x, t)
    mean = many.train_epoch(order, b, 1e-3)
    assert mean == np.float32(sum(float(v) for v in losses) / 10)
    assert np.array_equal(one.get_params().view(np.int32), many.get_params().view(np.int32))
