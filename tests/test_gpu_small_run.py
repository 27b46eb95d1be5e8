"""Transitions of small models in one launch (fp32, up to four chains, X in the
registers of a workgroup) at the edges of its layouts, against the FP64 oracle."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu

# columns on both sides of 4, 8, 16 and up to 32; rows on both sides of each
# multiple of 1024 and the most that fit (8192, 4096, 2048, 1024)
SHAPES = [(1, 1, 1), (17, 3, 4), (1024, 4, 2), (1025, 4, 1), (2049, 2, 3), (8192, 4, 1),
          (4096, 5, 2), (2050, 8, 1), (1000, 10, 1), (2048, 16, 4), (1025, 9, 2), (1024, 32, 1),
          (63, 17, 3)]


@pytest.mark.parametrize('lik', ['bernoulli', 'normal'])
@pytest.mark.parametrize('N,D,C', SHAPES)
def test_small_run(N, D, C, lik):
  """Three transitions with device randomness against the oracle driven by
  the same Philox draws: positions within 1e-4 relative (fp32 gradients over
  18 leapfrog steps; three orders above a rounding).  The same draws fed one
  transition at a time, the counts, the moments and the state."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d C=%d %s' % (N, D, C, lik), flush=True)
  rng = np.random.default_rng(13)
  X = rng.normal(size=(N, D)).astype(np.float32)
  w = rng.normal(size=D) * 0.3 / np.sqrt(D)
  y = (rng.random(N) < 1.0 / (1.0 + np.exp(-X @ w))).astype(np.float32)
  W0 = (w + 0.1 * rng.normal(size=(C, D))).astype(np.float32)
  loc, scale = 0.1 * rng.normal(size=D), 0.5 + rng.random(D)
  eps, L, T, seed = 0.2 / np.sqrt(N + 4.0), 6, 3, 5
  eng = GLMEngine(X, y, loc, scale, likelihood=lik)
  eng.set_state(W0)
  eng.moments_enable()
  params = torch.empty(T + 1, C, D, device='cuda')
  n_acc = torch.zeros(C, dtype=torch.int32, device='cuda')
  eng.run(params, eps, L, t0=1, n_iter=T, seed=seed, counter0=2, n_accept=n_acc)
  z_end, lp_end, g_end = eng.get_state()
  mean, _, n = eng.moments()
  m = O.GLM(X.astype(np.float64), y, loc.astype(np.float32).astype(np.float64),
            scale.astype(np.float32).astype(np.float64), likelihood=lik)
  z, acc = W0.astype(np.float64), np.zeros(C, int)
  for t in range(T):
    out = O.hmc_transition(z, O.momentum_normals(seed, 3 + t, C, D),
                           O.accept_uniforms(seed, 3 + t, C), float(np.float32(eps)), L,
                           m.logp_grad)
    z = out['z']
    acc += out['accept']
    got = params[1 + t].cpu().numpy()
    err = np.linalg.norm(got - z, axis=1) / np.linalg.norm(z, axis=1)
    assert err.max() < 1e-4, (t, err)
  assert np.array_equal(n_acc.cpu().numpy(), acc)
  assert n == T
  np.testing.assert_allclose(mean.cpu().numpy(), params[1:].double().mean(0).cpu().numpy(),
                             rtol=1e-12, atol=1e-14)
  assert torch.equal(z_end, params[T])
  lp_ref, g_ref = m.logp_grad(z_end.cpu().numpy().astype(np.float64))
  # sums of N fp32 terms of order 1: some 1e-6 of their absolute sum at most
  assert (np.abs(lp_end.cpu().numpy() - lp_ref) <= 1e-6 * (np.abs(lp_ref) + N + D)).all()
  assert (np.abs(g_end.cpu().numpy() - g_ref) <= 1e-5 * (N + np.abs(g_ref)) + 1e-5).all()
  # fed one at a time: the same bits
  eng.set_state(W0)
  one = torch.empty(C, D, device='cuda')
  for t in range(T):
    eng.transition(eps, L, momenta=eng.draw_momenta(C, seed, 3 + t),
                   uniforms=eng.draw_uniforms(C, seed, 3 + t), sample_out=one)
    assert torch.equal(one, params[1 + t]), t
