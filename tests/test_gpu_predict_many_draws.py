"""The fp32 posterior predictive of thousands of draws: fewer row ranges than
XCDs, as many on each, and more than run together, against FP64."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu

# one range, two and seven (of 128 rows), eight and more; draws whose tiles
# leave a round of ranges full, part empty, and more than full
SHAPES = [(100, 20, 3000), (200, 250, 3000), (896, 60, 2000), (897, 60, 2000), (3000, 250, 3000),
          (2500, 200, 5000), (1500, 130, 10000), (1100, 10, 20000), (5001, 100, 7001)]


@pytest.mark.parametrize('N,D,S', SHAPES)
def test_many_draws(N, D, S):
  """Log-likelihood: fp32 terms (eta within 1e-6 of sum |w x|, each term 6e-8
  relative) summed in FP64.  Mean response: partial sums of 32 fp32 values,
  added in FP64, each within eta's error.  The log-likelihood of the pass with
  replicates, whose eta has the same bits, agrees to FP64 rounding."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d S=%d' % (N, D, S), flush=True)
  g = torch.Generator(device='cuda').manual_seed(N + S)
  X = torch.randn(N, D, generator=g, device='cuda')
  w = torch.randn(D, generator=g, device='cuda') / D ** 0.5
  y = (torch.rand(N, generator=g, device='cuda') < torch.sigmoid(X @ w)).float()
  W = w + 0.1 * torch.randn(S, D, generator=g, device='cuda')
  eng = GLMEngine(X, y)
  mean, ll, _ = eng.predict(W)
  Wd, Xd, yd = (v.cpu().numpy().astype(np.float64) for v in (W, X, y))
  eta = Wd @ Xd.T
  d_eta = 1e-6 * (np.abs(Wd) @ np.abs(Xd).T)
  mu = O.sigmoid(eta)
  t = yd * eta - O.softplus(eta)
  bar = (np.abs(yd - mu) * d_eta).sum(1) + 1e-6 * np.abs(t).sum(1) + 1e-6
  assert (np.abs(ll.cpu().numpy() - t.sum(1)) <= bar).all()
  bar = 0.25 * d_eta.mean(0) + 1e-6 + 6e-8 * 32 * np.abs(mu).mean(0) + 1e-6
  assert (np.abs(mean.cpu().numpy() - mu.mean(0)) <= bar).all()
  m2, ll2, _ = eng.predict(W, replicate=True, seed=1)
  np.testing.assert_allclose(ll.cpu().numpy(), ll2.cpu().numpy(), rtol=1e-12)
