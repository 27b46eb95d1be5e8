"""The least-squares start of the surrogate's linear skip: Gram products at
the edges of their 64-column blocks, 32-row stages and row splits, and the
positive definite solve at the edges of its 32-row panels, against FP64."""

import numpy as np
import pytest
import torch

from edward_amd import _lib as L

pytestmark = pytest.mark.gpu


def _engine(D):
  from edward_amd.engine import GLMEngine
  from edward_amd.surrogate import Surrogate
  eng = GLMEngine(np.ones((64, D), np.float32), np.ones(64, np.float32), precision='bf16')
  return eng, Surrogate(eng, hidden=64, max_batch=64)


def _gram(eng, W, G, idx):
  D = W.shape[1]
  a = torch.empty(D, D, dtype=torch.float64, device='cuda')
  b = torch.empty_like(a)
  eng.check(eng.lib.edhmc_sur_skip_gram(eng.h, L.ptr(W), L.ptr(G), W.shape[0], L.ptr(idx),
                                        len(idx), L.ptr(a), L.ptr(b), eng.stream))
  return a, b


@pytest.mark.parametrize('offset', [0, 1])
@pytest.mark.parametrize('n,D', [(1, 1), (31, 4), (33, 63), (127, 64), (129, 65), (1000, 8),
                                 (4097, 130), (2500, 256), (9001, 300), (700, 511)])
def test_skip_gram(n, D, offset):
  """x and t in fp32 as the kernel forms them, the sums in FP64: at most n
  roundings of 1.1e-16 of the terms' absolute sum, below 1e-12 of it.  offset:
  rows that are not 16-byte aligned.  Two calls bit for bit; a captured call
  (one split) replayed three times within the same bound."""
  print('case n=%d D=%d offset=%d' % (n, D, offset), flush=True)
  rng = np.random.default_rng(5)
  P = 3 * n // 2 + 1
  eng, sur = _engine(D)
  W, G = [torch.from_numpy(rng.normal(size=P * D + 1).astype(np.float32)).cuda()
          [offset:offset + P * D].view(P, D) for _ in range(2)]
  nrm = [rng.normal(size=D), 0.5 + rng.random(D), rng.normal(size=D), 0.5 + rng.random(D)]
  sur.set_normalisation(*nrm)
  sel = rng.integers(0, P, size=n)
  idx = torch.from_numpy(sel).cuda()
  a, b = _gram(eng, W, G, idx)
  a2, b2 = _gram(eng, W, G, idx)
  assert torch.equal(a, a2) and torch.equal(b, b2)
  f = [v.astype(np.float32) for v in nrm]
  x = ((W.cpu().numpy()[sel] - f[0]) * f[1]).astype(np.float64)
  t = ((G.cpu().numpy()[sel] - f[2]) / f[3]).astype(np.float64)
  bar_a, bar_b = 1e-12 * (np.abs(x).T @ np.abs(x)), 1e-12 * (np.abs(x).T @ np.abs(t))
  assert (np.abs(a.cpu().numpy() - x.T @ x) <= bar_a).all()
  assert (np.abs(b.cpu().numpy() - x.T @ t) <= bar_b).all()
  side = torch.cuda.Stream()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph, stream=side):
    a3, b3 = _gram(eng, W, G, idx)
  for _ in range(3):
    a3.zero_()
    b3.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert (np.abs(a3.cpu().numpy() - x.T @ x) <= bar_a).all()
    assert (np.abs(b3.cpu().numpy() - x.T @ t) <= bar_b).all()


def test_skip_gram_bad_index():
  eng, sur = _engine(70)
  sur.set_normalisation(*[np.ones(70)] * 4)
  W = torch.randn(500, 70, device='cuda')
  for bad in (-1, 500):
    idx = torch.arange(500, device='cuda')
    idx[301] = bad
    a, b = _gram(eng, W, W, idx)
    assert torch.isnan(a).all() and torch.isnan(b).all()


@pytest.mark.parametrize('n', [1, 5, 31, 32, 33, 100, 256, 513])
def test_solve_spd(n):
  """Against LAPACK in FP64; the result is rounded to fp32 (6e-8 relative) and
  both solves lose at most the condition number (below 1e3 here) times
  1e-16 n: within 1e-7 of the largest entry."""
  rng = np.random.default_rng(n)
  eng, _ = _engine(8)
  M = rng.normal(size=(n, 3 * n))
  A, B, ridge = M @ M.T, rng.normal(size=(n, n)), 0.1 * n
  dA, dB = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
  xt = torch.empty(n, n, device='cuda')
  bad = torch.empty(1, dtype=torch.int32, device='cuda')
  work = torch.empty(eng.lib.edhmc_solve_spd_work(n), dtype=torch.uint8, device='cuda')

  def solve(dA):
    eng.check(eng.lib.edhmc_solve_spd(eng.h, L.ptr(dA), L.ptr(dB), n, ridge, L.ptr(xt),
                                      L.ptr(bad), L.ptr(work), eng.stream))
    return int(bad.item())
  assert solve(dA) == 0
  ref = np.linalg.solve(A + ridge * np.eye(n), B).T
  assert np.abs(xt.cpu().numpy() - ref).max() <= 1e-7 * np.abs(ref).max()
  for v in (-1e9, float('nan')):
    dA2 = dA.clone()
    dA2[n // 2, n // 2] = v
    assert solve(dA2) == 1


def test_singular_start_raises():
  """A constant coordinate and no ridge: the general solve's error."""
  eng, sur = _engine(6)
  W = torch.randn(100, 6, device='cuda')
  W[:, 2] = 1.0
  G = torch.randn(100, 6, device='cuda')
  sur.normalise_from(W, G)
  with pytest.raises(np.linalg.LinAlgError):
    sur.init_skip_least_squares(W, G, ridge=0.0)
