"""The radiance cache's training step at the edges of its split: tiles of 64
records over the blocks (one of 1, 63 and 64 records, a ragged last one) and
gradient rows over 16 waves (fewer than 16 rows, 16, 17, and several each),
against the FP64 oracle and the FP64 sum of the rows.

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
