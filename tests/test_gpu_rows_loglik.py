"""The order in which the one-pass fp32 gradient sums the log-likelihood's FP64
terms: that of the two-product form, whatever the row ranges.  A log ratio is
the difference of two such sums, so their last bits show."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _tree_sum(t):
  """t [N] by 128-row tiles (bits 5 4 3 2 1 0 of the row, then the two
  halves), the tiles in 16 runs of four interleaved strides each."""
  n_tiles = -(-len(t) // 256) * 2
  x = np.zeros(n_tiles * 128)
  x[:len(t)] = t
  x = x.reshape(n_tiles, 2, 64)
  while x.shape[2] > 1:
    half = x.shape[2] // 2
    x = x[:, :, :half] + x[:, :, half:]
  tiles = x[:, 0, 0] + x[:, 1, 0]
  per = -(-n_tiles // 16)
  total = 0.0
  for k in range(16):
    run = tiles[k * per:(k + 1) * per]
    part = [0.0] * 4
    for i, v in enumerate(run):
      part[i % 4] += v
    total += ((part[0] + part[1]) + part[2]) + part[3]
  return total


# ranges of 128 rows and more that divide no tile, a tile of padding, one range;
# chains for the column-split form in both its widths and for the chain-split one
@pytest.mark.parametrize('N,D,C', [(257, 3, 7), (1000, 64, 40), (9001, 100, 30),
                                   (20011, 50, 449), (9000, 190, 700), (5003, 256, 513),
                                   (40000, 20, 300), (65537, 130, 520), (3000, 60, 1030)])
def test_loglik_order(N, D, C):
  """Normal likelihood.  Positions and data are dyadic with so few bits that
  eta is exact in fp32, and y - eta, its square and the FP64 term round once
  each in numpy as on the device: the sum has the same bits.  The prior's sum
  (some 1e-13) is far below half a unit in the last place of the log joint;
  it may still tip a rounding: one unit is allowed on a hundredth of the
  chains, none beyond."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d C=%d' % (N, D, C), flush=True)
  rng = np.random.default_rng(41)
  X = (rng.integers(-16, 17, size=(N, D)) / 8.0).astype(np.float32)
  W = (rng.integers(-8, 9, size=(C, D)) / 16.0).astype(np.float32)
  y = (6.0 * rng.normal(size=N)).astype(np.float32)
  eng = GLMEngine(X, y, likelihood='normal', lik_scale=1.0)
  lp, _ = eng.logp_grad(W)
  lp = lp.cpu().numpy()
  prior = (-0.5 * W.astype(np.float64) ** 2 - 0.5 * np.log(2 * np.pi)).sum(1)
  cs = np.unique(np.concatenate([rng.integers(0, C, size=100), [0, C - 1]]))
  off = 0
  for c in cs:
    eta = (X.astype(np.float64) @ W[c].astype(np.float64)).astype(np.float32)
    d = y - eta
    t = -0.5 * (d * d).astype(np.float64) - 0.5 * np.log(2 * np.pi)
    want = _tree_sum(t) + prior[c]
    assert abs(lp[c] - want) <= np.spacing(abs(want)), (c, lp[c], want)
    off += lp[c] != want
  assert off <= max(1, len(cs) // 100)
  lp2, _ = eng.logp_grad(W)
  assert np.array_equal(lp, lp2.cpu().numpy())
