"""The one-pass fp32 gradient (D_pad <= 256, five chains and more) at the
edges of its row tiles, row ranges and chain blocks, in both its forms (few
chains: columns split over the waves; many: chains), against FP64."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu

# rows around 16, 32, 64 and the ranges' ends; columns in each multiple of 64;
# chains around 16, 32, 64 and around the change of form (512 with 64 ranges)
SHAPES = [(1, 1, 5), (15, 64, 16), (17, 65, 17), (63, 130, 33), (65, 250, 31), (257, 193, 64),
          (1000, 100, 65), (1025, 64, 200), (4111, 192, 129), (9001, 256, 100),
          (20011, 50, 449), (20000, 128, 448), (9000, 190, 700), (5003, 256, 513),
          (12345, 60, 1030), (3000, 127, 640)]


@pytest.mark.parametrize('lik', ['bernoulli', 'normal'])
@pytest.mark.parametrize('N,D,C', SHAPES)
def test_rows_terms(N, D, C, lik):
  """Log joint and gradient.  A gradient entry sums N terms r x in fp32: its
  error is within 1e-6 of sum |r x| (fp32 rounding 6e-8 times the square root
  of a run, with eta's own rounding beside it); the log joint sums fp32 terms
  (6e-8 relative each) in FP64: within 1e-6 of the terms' absolute sum.  Two
  evaluations bit for bit."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d C=%d %s' % (N, D, C, lik), flush=True)
  rng = np.random.default_rng(17)
  X = rng.normal(size=(N, D)).astype(np.float32)
  w = rng.normal(size=D) * 0.3 / np.sqrt(D)
  y = (rng.random(N) < 1.0 / (1.0 + np.exp(-X @ w))).astype(np.float32)
  W0 = (w + 0.1 * rng.normal(size=(C, D))).astype(np.float32)
  s = 0.8
  eng = GLMEngine(X, y, likelihood=lik, lik_scale=s)
  lp, g = eng.logp_grad(W0)
  lp2, g2 = eng.logp_grad(W0)
  assert torch.equal(lp, lp2) and torch.equal(g, g2)
  Wd, Xd, yd = W0.astype(np.float64), X.astype(np.float64), y.astype(np.float64)
  eta = Wd @ Xd.T
  if lik == 'bernoulli':
    r = yd - O.sigmoid(eta)
    ll = yd * eta - O.softplus(eta)
  else:
    r = (yd - eta) / s ** 2
    ll = -0.5 * ((yd - eta) / s) ** 2 - np.log(s) - 0.5 * np.log(2 * np.pi)
  prior = -0.5 * Wd ** 2 - 0.5 * np.log(2 * np.pi)
  bar_g = 1e-6 * (np.abs(r) @ np.abs(Xd) + np.abs(Wd)) + 1e-6
  bar_l = 1e-6 * (np.abs(ll).sum(1) + np.abs(prior).sum(1)) + 1e-6
  assert (np.abs(g.cpu().numpy() - (r @ Xd - Wd)) <= bar_g).all()
  assert (np.abs(lp.cpu().numpy() - (ll.sum(1) + prior.sum(1))) <= bar_l).all()


# group sizes: groups that end on and beside the 16-row blocks, runs of single
# rows (several groups in a block), empty ones, groups across row ranges, one
# group that is nearly all of the data
_G = np.random.default_rng(29)
GROUPS = [
    [16, 32, 1, 15, 0, 17, 48, 0, 0, 3, 64],
    [1] * 70 + [0] * 5 + [2] * 33,
    list(_G.poisson(40, size=200)),
    [3, 6001, 1, 0, 2],
    list(_G.integers(0, 9, size=900)),
    list(_G.integers(100, 700, size=21)),
]


@pytest.mark.parametrize('D,C', [(5, 7), (64, 48), (100, 130), (30, 600), (130, 530)])
@pytest.mark.parametrize('k', range(len(GROUPS)))
def test_rows_groups(k, D, C):
  """Intercepts and group sums with few chains (sums in their own kernel) and
  many (within the gradient's walk over the rows).  A group's entry sums its
  rows' residuals in fp32, |r| <= 1 with eta's rounding: within 1e-6 of the
  group's size (+ 1e-6 of the prior's terms); w's entries as for the GLM.
  Two evaluations bit for bit."""
  from edward_amd.hier import HierEngine
  sizes = np.asarray(GROUPS[k])
  off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
  N, G = int(off[-1]), len(sizes)
  print('case %d N=%d G=%d D=%d C=%d' % (k, N, G, D, C), flush=True)
  rng = np.random.default_rng(31)
  X = rng.normal(size=(N, D)).astype(np.float32)
  group = np.repeat(np.arange(G), sizes)
  y = (rng.random(N) < 0.5).astype(np.float32)
  th = (rng.normal(size=(C, G + 2 + D)) * 0.3).astype(np.float32)
  eng = HierEngine(X, y, off)
  lp, g = eng.logp_grad(th)
  lp2, g2 = eng.logp_grad(th)
  assert torch.equal(lp, lp2) and torch.equal(g, g2)
  m = O.HierLogReg(X.astype(np.float64), y, off)
  lp_ref, g_ref = m.logp_grad(th.astype(np.float64))
  td, Xd = th.astype(np.float64), X.astype(np.float64)
  r = y - O.sigmoid(td[:, group] + td[:, G + 2:] @ Xd.T)
  tau = np.exp(-2 * td[:, G + 1])[:, None]
  d = np.abs(td[:, :G] - td[:, G:G + 1])
  bar = np.empty_like(td)
  bar[:, :G] = sizes + d * tau
  bar[:, G] = (d * tau).sum(1) + 1
  bar[:, G + 1] = (d * d * tau).sum(1) + G + 1
  bar[:, G + 2:] = np.abs(r) @ np.abs(Xd) + 1
  assert (np.abs(g.cpu().numpy() - g_ref) <= 1e-6 * bar + 1e-6).all()
  assert (np.abs(lp.cpu().numpy() - lp_ref) <= 1e-6 * np.abs(lp_ref) + 1e-3).all()
