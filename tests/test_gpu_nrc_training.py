"""The radiance cache's training step at the edges of its split: tiles of 64
records over the blocks (one of 1, 63 and 64 records, a ragged last one) and
gradient rows over 16 waves (fewer than 16 rows, 16, 17, and several each),
against the FP64 oracle and the FP64 sum of the rows, and the fp32 sums bit
for bit against their order.

Tolerances: as test_gpu_nrc.py for the gradients (bf16 storage against the
oracle's bf16 roundings: 2 % relative L2 per layer, losses 0.5 %); a sum of
t rows in fp32, in any order, is within t 2^-24 sum |row| of the exact one,
and the moment's product adds two roundings.
"""
import numpy as np
import pytest

from oracle import nrc_ref as R
from test_gpu_nrc import Net, _bf16_dev, _features

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 16 * 64, 16 * 64 + 1, 41 * 64 - 7])
def test_training_step_of_any_length(n):
    net = Net()
    params = R.init_params(21)
    net.set_params(params)
    x = _features(n, 22)
    t = np.random.default_rng(23).uniform(0, 1, (n, 3))
    loss, g = net.train(_bf16_dev(x), t)
    want_loss, want = R.loss_and_grad(params, x, t, bf16=True)
    assert abs(loss - want_loss) <= 5e-3 * want_loss, (loss, want_loss)
    for i in range(5):
        a, b = R.OFFSETS[i], R.OFFSETS[i + 1]
        assert np.linalg.norm(g[a:b] - want[a:b]) <= 2e-2 * np.linalg.norm(want[a:b]), i
    tiles = (n + 63) // 64
    rows = net.partial.view(-1, R.N_PARAMS).cpu().numpy().astype(np.float64)
    assert np.all(rows[tiles:] == 0)  # nothing past the last tile's row
    net.adam(n, 1e-2, 1)
    m, mag = net.m.cpu().numpy().astype(np.float64), np.abs(rows).sum(0)
    assert np.all(np.abs(m - 0.1 * rows.sum(0)) <= 0.1 * (tiles + 2) * 2.0 ** -24 * mag + 1e-45)
    tl = net.tile_loss[:tiles].cpu().numpy().astype(np.float64)
    assert abs(float(net.loss.item()) - tl.sum()) <= tiles * 2.0 ** -24 * tl.sum()


@pytest.mark.parametrize("n", [1, 63, 17 * 64 + 1, 257 * 64 + 1])
def test_sums_keep_their_order(n):
    """A step gives the same bits whatever its split over waves: the loss of a
    tile, the sum of the tiles' losses and the sums of the gradient rows are
    those of one fixed order in fp32, and the inference that the loss is
    recomputed from adds in the training kernel's order."""
    f = np.float32
    tiles = (n + 63) // 64
    net = Net(max_tiles=tiles)
    net.set_params(R.init_params(41))
    x = _bf16_dev(_features(n, 42))
    t = np.random.default_rng(43).uniform(0, 1, (n, 3)).astype(f)
    net.train(x, t)
    y = np.zeros((tiles * 64, 3), f)
    y[:n] = net.infer(x)
    term = np.zeros((tiles * 64, 3), f)
    d = y[:n] - t
    term[:n] = d * d / (y[:n] * y[:n] + f(0.01)) * (f(1) / (f(3) * f(n)))
    lane = np.zeros((tiles, 16), f)  # query 16 k + r is lane r's
    for k in range(4):
        for c in range(3):
            lane += term.reshape(tiles, 64, 3)[:, 16 * k:16 * k + 16, c]
    for o in (8, 4, 2, 1):
        lane = lane + lane[:, np.arange(16) ^ o]
    assert np.array_equal(net.tile_loss.cpu().numpy(), lane[:, 0])
    rows = net.partial.view(tiles, R.N_PARAMS).cpu().numpy()
    net.adam(n, 1e-2, 1)
    group = np.zeros((4, R.N_PARAMS), f)
    loss = f(0)
    for k in range(tiles):
        group[k % 4] += rows[k]
        loss += lane[k, 0]
    g = (group[0] + group[1]) + (group[2] + group[3])
    assert np.array_equal(net.m.cpu().numpy(), f(0.9) * np.zeros_like(g) + f(0.1) * g)
    assert net.loss.item() == loss
