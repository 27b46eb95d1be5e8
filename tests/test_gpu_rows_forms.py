"""The two forms of the one-pass fp32 gradient give a chain the same bits: the
chain-split one stands in where the other's memory does not fit."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# 256 chains take the column-split form and 512 the other, over the same ranges
# of rows; rows that divide nothing, ranges that divide no tile
@pytest.mark.parametrize('N,D', [(70001, 60), (70001, 128), (40011, 190), (33333, 250)])
def test_glm(N, D):
  from edward_amd.engine import GLMEngine
  print('case N=%d D=%d' % (N, D), flush=True)
  g = torch.Generator(device='cuda').manual_seed(N + D)
  X = torch.randn(N, D, generator=g, device='cuda')
  y = (torch.rand(N, generator=g, device='cuda') < 0.5).float()
  W = 0.1 * torch.randn(512, D, generator=g, device='cuda')
  eng = GLMEngine(X, y)
  lw, gw = eng.logp_grad(W)
  ln, gn = eng.logp_grad(W[:256].contiguous())
  assert torch.equal(gw[:256], gn) and torch.equal(lw[:256], ln)


@pytest.mark.parametrize('G,m,D', [(700, 100, 60), (9, 8000, 20), (5000, 14, 128), (3, 23333, 200)])
def test_hierarchical(G, m, D):
  """Group sums, kept within the pass by one form and left to a kernel of their
  own by the other, included."""
  from edward_amd.hier import HierEngine
  print('case G=%d m=%d D=%d' % (G, m, D), flush=True)
  rng = np.random.default_rng(G)
  sizes = rng.poisson(m, size=G)
  sizes[G // 2] = 0
  off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int64)
  N = int(off[-1])
  g = torch.Generator(device='cuda').manual_seed(G + D)
  X = torch.randn(N, D, generator=g, device='cuda')
  y = (torch.rand(N, generator=g, device='cuda') < 0.5).float()
  th = 0.1 * torch.randn(512, G + 2 + D, generator=g, device='cuda')
  eng = HierEngine(X, y, off)
  lw, gw = [v.clone() for v in eng.logp_grad(th)]
  ln, gn = eng.logp_grad(th[:256].contiguous())
  assert torch.equal(gw[:256], gn) and torch.equal(lw[:256], ln)
