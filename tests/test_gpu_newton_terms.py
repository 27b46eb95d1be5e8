"""Newton terms at the edges of the Gram kernel's blocks (64, 128 and 256
columns), stages and row slices, against FP64."""

import numpy as np
import pytest
import torch

from oracle import hmc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['fp32', 'bf16'])
@pytest.mark.parametrize('N,D', [(1, 1), (7, 64), (63, 65), (64, 130), (65, 256), (2049, 255),
                                 (4097, 192), (8200, 300), (6145, 512), (5000, 640),
                                 (3001, 700), (2100, 1024)])
def test_newton_terms_edges(N, D, precision):
  """Each entry of the negative Hessian sums N fp32 terms s x_i x_j in 64
  chains (rounding 6e-8 times the square root of a chain, the factor s x_i
  rounded too): within 1e-6 of the terms' absolute sum, plus the prior's; the
  gradient likewise with r; the log joint sums FP64 terms whose eta carries
  fp32 rounding: within 1e-6 of their absolute sum."""
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d %s' % (N, D, precision), flush=True)
  rng = np.random.default_rng(3)
  X = rng.normal(size=(N, D)).astype(np.float32)
  if precision == 'bf16':
    X = torch.from_numpy(X).bfloat16().float().numpy()
  y = (rng.random(N) < 0.5).astype(np.float32)
  w = (rng.normal(size=D) / np.sqrt(D)).astype(np.float32)
  eng = GLMEngine(X, y, precision=precision)
  lp, g, P = eng.newton_terms(w)
  Xd, wd = X.astype(np.float64), w.astype(np.float64)
  eta = Xd @ wd
  sig = O.sigmoid(eta)
  r, s = y - sig, sig * (1.0 - sig)
  ll = y * eta - O.softplus(eta)
  prior = -0.5 * wd ** 2 - 0.5 * np.log(2 * np.pi)
  aX = np.abs(Xd)
  assert (np.abs(P - ((Xd * s[:, None]).T @ Xd + np.eye(D)))
          <= 1e-6 * ((aX * s[:, None]).T @ aX + np.eye(D))).all()
  assert (np.abs(g - (r @ Xd - wd)) <= 1e-6 * (np.abs(r) @ aX + np.abs(wd)) + 1e-6).all()
  assert abs(lp - (ll.sum() + prior.sum())) <= 1e-6 * (np.abs(ll).sum() + np.abs(prior).sum())
