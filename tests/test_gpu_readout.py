"""Readout kernels (column moments, autocovariances) against FP64 numpy."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# draws, chains, coordinates around the kernels' edges: single columns, fewer
# columns than a wave, rows per thread of 8 and 32 and beyond, lag blocks of
# 32 and steps of 8, columns just past a strip of 64
SHAPES = [(2, 1, 1), (5, 3, 2), (7, 70, 3), (33, 2, 65), (100, 130, 1), (129, 5, 64),
          (1000, 9, 64), (2048, 2, 20), (2049, 3, 43), (9000, 1, 10)]


def _store(T, C, D):
  rng = np.random.default_rng(T + C + D)
  x = rng.normal(size=(T, C, D))
  for t in range(1, T):
    x[t] += 0.7 * x[t - 1]
  return (x + 3.0 * rng.normal(size=(1, C, D))).astype(np.float32)


@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
@pytest.mark.parametrize('T,C,D', SHAPES)
def test_moments(T, C, D, dtype):
  """FP64 two-pass sums of T terms: 1e-13 relative is some hundred roundings
  (2^-53) for the variance, and for the mean relative to the terms."""
  from edward_amd import readout
  x = _store(T, C, D)
  for burn in (0, T // 3):
    mean, var = readout.empirical_moments(torch.as_tensor(x, device='cuda').to(dtype), burn)
    a = x.astype(np.float64)[burn:]
    np.testing.assert_allclose(mean.cpu().numpy(), a.mean(0), rtol=1e-13,
                               atol=1e-13 * np.abs(a).max())
    np.testing.assert_allclose(var.cpu().numpy(), a.var(0), rtol=1e-13, atol=1e-30)


@pytest.mark.parametrize('T,C,D', SHAPES)
def test_autocov(T, C, D):
  """Every lag in one window and in two pieces: the FP64 sum of up to T C
  products, error within 1e-13 of the lag-0 sum (their Cauchy-Schwarz
  bound)."""
  from edward_amd import diagnostics
  from edward_amd.engine import Context
  x = _store(T, C, D)
  s = torch.as_tensor(x, device='cuda')
  eng = Context()
  top = min(T - 1, 400)
  acov, cmean = diagnostics.autocov(eng, s, top)
  a = x.astype(np.float64)
  a = a - a.mean(0)
  ref = np.stack([(a[:T - l] * a[l:]).sum((0, 1)) / T for l in range(top + 1)])
  bar = 1e-13 * ref[0] + 1e-300
  np.testing.assert_allclose(cmean.cpu().numpy(), x.astype(np.float64).mean(0), rtol=1e-12)
  assert (np.abs(acov.cpu().numpy() - ref) <= bar).all()
  cut = top // 2 + 1
  if cut <= top:
    more = diagnostics.autocov_lags(eng, s, cut, top + 1 - cut, cmean)
    assert (np.abs(more.cpu().numpy() - ref[cut:]) <= bar).all()
