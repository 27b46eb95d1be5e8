"""Autocovariances and effective sample sizes of many chains over few draws:
partial sums of many groups of chains, against FP64 numpy."""

import numpy as np
import pytest
import torch

from edward_amd import diagnostics as dg

pytestmark = pytest.mark.gpu


def _store(T, C, D):
  g = torch.Generator(device='cuda').manual_seed(T + C + D)
  s = torch.randn(T, C, D, generator=g, device='cuda')
  for t in range(1, T):
    s[t] += 0.6 * s[t - 1]
  return s + torch.randn(D, generator=g, device='cuda')


# draws around the last whose means come with the sums (64); lags around the
# two widths (8, 32) and those that take transforms; chains in one, several and
# hundreds of groups, side by side and not
@pytest.mark.parametrize('C,D', [(1, 1), (3, 70), (65, 1), (130, 33), (700, 10), (2500, 3)])
@pytest.mark.parametrize('T', [4, 9, 33, 64, 65, 150])
def test_few_draws(T, C, D):
  """Sums of C T products, in whatever order: every lag within 1e-13 of the
  lag-0 sum (2^-53 a rounding, some hundred of them in a row at most)."""
  from edward_amd.engine import Context
  print('case T=%d C=%d D=%d' % (T, C, D), flush=True)
  eng = Context()
  s = _store(T, C, D)
  x = s.double().cpu().numpy()
  a = x - x.mean(0)
  ref = np.stack([(a[:T - l] * a[l:]).sum((0, 1)) / T for l in range(T)])
  for lag in (0, 7, 8, 31, 32, T - 1):
    if lag >= T:
      continue
    acov, cmean = dg.autocov(eng, s, lag)
    assert (np.abs(acov.cpu().numpy() - ref[:lag + 1]) <= 1e-13 * ref[0]).all(), lag
    np.testing.assert_allclose(cmean.cpu().numpy(), x.mean(0), rtol=1e-12, atol=1e-13)
  np.testing.assert_allclose(dg.ess(eng, s), dg.ess_from_acov(ref, x.mean(0), T, True),
                             rtol=max(1e-10, 20 * T * 1e-13))


@pytest.mark.parametrize('T,lag', [(32, 5), (64, 63)])
def test_many_chains_in_parallel(T, lag):
  """Sixty-four times the chains (10 MB instead of 160 KB) take a few times as
  long, not one load after the other: 40 times as long where each lag and
  coordinate summed its groups of chains alone."""
  from edward_amd.engine import Context
  eng = Context()
  best = []
  for C in (64, 4096):
    s = _store(T, C, 10)
    times = []
    for _ in range(30):
      a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      a.record()
      for _ in range(5):
        dg.autocov(eng, s, lag)
      b.record()
      b.synchronize()
      times.append(a.elapsed_time(b))
    best.append(min(times))
  print('times', best, flush=True)
  assert best[1] < 12 * best[0], best
