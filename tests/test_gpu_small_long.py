"""Long runs of small models (fp32, up to four chains): one step a transition,
and more steps than one launch takes, against single transitions fed the same
draws."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# one launch takes max(1, 4096 / L) transitions
@pytest.mark.parametrize('L,T', [(1, 1000), (1, 4100), (2, 2050), (64, 130), (4097, 2)])
@pytest.mark.parametrize('N,D,C,lik', [(1500, 7, 3, 'bernoulli'), (90, 3, 1, 'normal')])
def test_long_run(N, D, C, lik, L, T):
  """Same draws, same arithmetic: the same bits, whatever the launches."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d C=%d %s L=%d T=%d' % (N, D, C, lik, L, T), flush=True)
  rng = np.random.default_rng(11)
  X = rng.normal(size=(N, D)).astype(np.float32)
  y = (rng.random(N) < 0.4).astype(np.float32)
  W0 = (0.1 * rng.normal(size=(C, D))).astype(np.float32)
  eps, seed = 0.9 / np.sqrt(0.25 * N) / L ** 0.5, 21
  eng = GLMEngine(X, y, likelihood=lik)

  def state():
    z, lp, g = eng.get_state()
    mean, var, n = eng.moments()
    assert n == T
    return z, lp, g, mean, var, eng.last_ratio()

  eng.set_state(W0)
  eng.moments_enable()
  params = torch.empty(T, C, D, device='cuda')
  n_acc = torch.zeros(C, dtype=torch.int32, device='cuda')
  eng.run(params, eps, L, seed=seed, n_accept=n_acc)
  got = state()

  eng.set_state(W0)
  eng.moments_enable()
  one = torch.empty(T, C, D, device='cuda')
  n_one = torch.zeros(C, dtype=torch.int32, device='cuda')
  for t in range(T):
    eng.transition(eps, L, momenta=eng.draw_momenta(C, seed, t),
                   uniforms=eng.draw_uniforms(C, seed, t), sample_out=one[t], n_accept=n_one)
  ref = state()
  same = (params == one).all(2)
  assert same.all(), 'chain and transition of the first difference: %s' % (
      torch.nonzero(~same)[0].tolist())
  assert torch.equal(n_acc, n_one) and 0 < int(n_acc.min())
  for a, b in zip(got, ref):
    assert torch.equal(torch.as_tensor(a), torch.as_tensor(b))
