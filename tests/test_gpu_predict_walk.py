"""The fp32 posterior predictive without replicates (D_pad <= 256) at the edges
of its tiles, row ranges and draw blocks, against FP64."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu

# columns in every count of 16-column chunks; rows around blocks, tiles, ranges;
# draws for one, two and four waves along them and for several tiles
SHAPES = [(1, 1, 1), (17, 16, 5), (64, 17, 64), (127, 33, 65), (129, 50, 100), (513, 65, 128),
          (1000, 81, 300), (4097, 100, 500), (900, 113, 250), (2000, 128, 64), (700, 129, 33),
          (1500, 161, 40), (999, 200, 129), (333, 256, 257), (70001, 20, 70)]


@pytest.mark.parametrize('lik', ['bernoulli', 'normal'])
@pytest.mark.parametrize('N,D,S', SHAPES)
def test_predict_walk(N, D, S, lik):
  """Log-likelihood: fp32 terms (eta within 1e-6 of sum |w x|, each term 6e-8
  relative) summed in FP64.  Mean response: an fp32 sum of S values, each
  within eta's error.  The log-likelihood of the pass with replicates, whose
  eta has the same bits, agrees to FP64 rounding."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d S=%d %s' % (N, D, S, lik), flush=True)
  rng = np.random.default_rng(23)
  X = rng.normal(size=(N, D)).astype(np.float32)
  w = rng.normal(size=D) / np.sqrt(D)
  y = (rng.random(N) < 1.0 / (1.0 + np.exp(-X @ w))).astype(np.float32)
  W = (w + 0.1 * rng.normal(size=(S, D))).astype(np.float32)
  eng = GLMEngine(X, y, likelihood=lik, lik_scale=0.8)
  mean, ll, _ = eng.predict(W)
  Wd, Xd, yd = W.astype(np.float64), X.astype(np.float64), y.astype(np.float64)
  eta = Wd @ Xd.T
  d_eta = 1e-6 * (np.abs(Wd) @ np.abs(Xd).T)
  if lik == 'bernoulli':
    t, slope, mu = yd * eta - O.softplus(eta), np.abs(yd - O.sigmoid(eta)), O.sigmoid(eta)
    d_mu = 0.25 * d_eta + 1e-6
  else:
    t = -0.5 * ((yd - eta) / 0.8) ** 2 - np.log(0.8) - 0.5 * np.log(2 * np.pi)
    slope, mu, d_mu = np.abs(yd - eta) / 0.64, eta, d_eta + 1e-6 * np.abs(eta)
  bar = (slope * d_eta).sum(1) + 1e-6 * np.abs(t).sum(1) + 1e-6
  assert (np.abs(ll.cpu().numpy() - t.sum(1)) <= bar).all()
  bar = d_mu.mean(0) + 6e-8 * np.sqrt(S) * np.abs(mu).mean(0) + 1e-6
  assert (np.abs(mean.cpu().numpy() - mu.mean(0)) <= bar).all()
  _, ll2, _ = eng.predict(W, replicate=True, seed=1)
  np.testing.assert_allclose(ll.cpu().numpy(), ll2.cpu().numpy(), rtol=1e-12)
  m3, ll3, _ = eng.predict(W)
  assert torch.equal(m3, mean) and torch.equal(ll3, ll)
