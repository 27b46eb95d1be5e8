"""The surrogate's weight and bias gradients in one launch each, with products
of unequal sizes and on both sides of the width (128 tiles of 128 x 128)
from which each product takes a launch of its own."""

import numpy as np
import pytest
import torch

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('D,H,B', [(1, 1, 1), (130, 129, 127), (60, 300, 257), (300, 60, 128),
                                   (20, 1408, 140), (20, 1409, 140)])
def test_weight_grads(D, H, B):
  """bf16 products (2^-9 a rounding, several of them per layer) against the
  FP64 oracle: 3e-2 of each gradient's norm; two evaluations bit for bit."""
  from edward_amd.engine import GLMEngine
  from edward_amd.surrogate import Surrogate
  print('case D=%d H=%d B=%d' % (D, H, B), flush=True)
  rng = np.random.default_rng(7)
  eng = GLMEngine(rng.normal(size=(300, D)).astype(np.float32), np.ones(300, np.float32),
                  precision='bf16')
  sur = Surrogate(eng, hidden=H, max_batch=B, seed=1)
  norm = {'in_shift': rng.normal(size=D) * 0.1, 'in_scale': rng.uniform(0.5, 2, size=D),
          'out_shift': rng.normal(size=D), 'out_scale': rng.uniform(0.5, 3, size=D)}
  sur.set_normalisation(*[norm[k].astype(np.float32) for k in
                          ('in_shift', 'in_scale', 'out_shift', 'out_scale')])
  W = rng.normal(size=(B, D)).astype(np.float32)
  G = (3 * rng.normal(size=(B, D))).astype(np.float32)
  _, grad = sur.loss_grad(torch.tensor(W), torch.tensor(G))
  _, grad2 = sur.loss_grad(torch.tensor(W), torch.tensor(G))
  assert torch.equal(grad, grad2)
  p = MO.unflatten(sur.get_params().cpu().numpy(), D, H)
  _, ref = MO.loss_and_grad(p, W.astype(np.float64), G.astype(np.float64), norm)
  got = MO.unflatten(grad.cpu().numpy(), D, H)
  for k in ('W1', 'b1', 'W2', 'b2', 'W3', 'b3'):
    d = np.linalg.norm(got[k] - ref[k])
    assert d <= 3e-2 * np.linalg.norm(ref[k]) + 1e-6, (k, d)
