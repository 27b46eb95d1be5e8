"""The few-chain gradient (fp32, one to four chains, D <= 256: one pass over X,
residuals in registers) against the FP64 oracle and against the two-kernel
pass that takes five chains and more."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu

# column counts around the layouts' edges (16, 32, 48 columns, then multiples
# of 64), rows around the tiles' (64, 128 or 256 rows) and the ranges'
SHAPES = [(1, 1, 1), (63, 16, 2), (64, 17, 4), (65, 33, 3), (257, 48, 1), (1000, 10, 1),
          (1025, 49, 4), (4099, 64, 2), (20000, 65, 1), (70001, 128, 4), (3001, 129, 3),
          (5000, 200, 1), (9001, 256, 4), (300007, 5, 2)]


def _problem(N, D, C, seed):
  rng = np.random.default_rng(seed)
  X = rng.normal(size=(N, D)).astype(np.float32)
  w = rng.normal(size=D) * 0.3 / np.sqrt(D)
  y = (rng.random(N) < 1.0 / (1.0 + np.exp(-X @ w))).astype(np.float32)
  W0 = (w + 0.1 * rng.normal(size=(C, D))).astype(np.float32)
  return X, y, W0, rng


@pytest.mark.parametrize('lik', ['bernoulli', 'normal'])
@pytest.mark.parametrize('N,D,C', SHAPES)
def test_few_chain_terms(N, D, C, lik):
  """Log joint and gradient at the layouts' edges.  A gradient entry sums N
  terms r x with |r| of order 1, in fp32 runs of at most N: error within
  1e-6 of sum |r x| per entry (fp32 rounding 6e-8 times the square root of
  the run, with eta's own rounding beside it); the log joint sums fp32 terms
  (6e-8 relative each) in FP64: within 1e-6 of the terms' absolute sum.  The
  forward-only log joint within the same of the gradient pass's; two
  evaluations bit for bit; rows of a call with four more chains (two-kernel
  pass) within twice the bar."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d C=%d %s' % (N, D, C, lik), flush=True)
  X, y, W0, _ = _problem(N, D, C, 7)
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
  g, lp = g.cpu().numpy(), lp.cpu().numpy()
  assert (np.abs(g - (r @ Xd - Wd)) <= bar_g).all()
  assert (np.abs(lp - (ll.sum(1) + prior.sum(1))) <= bar_l).all()
  assert (np.abs(eng.logp(W0).cpu().numpy() - lp) <= bar_l).all()
  lp4, g4 = eng.logp_grad(np.concatenate([W0, np.zeros((4, D), np.float32)]))
  assert (np.abs(g4.cpu().numpy()[:C] - g) <= 2 * bar_g).all()
  assert (np.abs(lp4.cpu().numpy()[:C] - lp) <= 2 * bar_l).all()


@pytest.mark.parametrize('N,D,C', [(1000, 10, 1), (5000, 54, 2), (20000, 100, 4)])
def test_few_chain_run(N, D, C):
  """A run of three transitions with device randomness against the oracle
  driven by the same Philox draws (positions within 1e-4 relative), twice
  with the same bits; the MH step of the same chains leaves a finite state."""
  from edward_amd.engine import GLMEngine
  X, y, W0, _ = _problem(N, D, C, 11)
  eps, L, T, seed = 0.3 / np.sqrt(N), 6, 3, 5
  eng = GLMEngine(X, y)
  outs = []
  for _ in range(2):
    eng.set_state(W0)
    params = torch.empty(T, C, D, device='cuda')
    eng.run(params, eps, L, seed=seed)
    outs.append(params.cpu().numpy())
  np.testing.assert_array_equal(outs[0], outs[1])
  m = O.GLM(X.astype(np.float64), y, np.zeros(D), np.ones(D))
  z = W0.astype(np.float64)
  for t in range(T):
    out = O.hmc_transition(z, O.momentum_normals(seed, t, C, D), O.accept_uniforms(seed, t, C),
                           float(np.float32(eps)), L, m.logp_grad)
    z = out['z']
    err = np.linalg.norm(outs[0][t] - z, axis=1) / np.linalg.norm(z, axis=1)
    assert err.max() < 1e-4, (t, err)
  eng.mh_step(0.001, seed=3, counter=1)
  assert all(torch.isfinite(v).all() for v in eng.get_state())
