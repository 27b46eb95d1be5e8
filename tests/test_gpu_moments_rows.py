"""Column moments of few rows: the two workgroup sizes at their border, against
FP64 numpy."""

import numpy as np
import pytest
import torch

from edward_amd import readout

pytestmark = pytest.mark.gpu


# 64 rows of 64 columns, 256 of 16 and 1024 of 4 are the most 256 threads hold
@pytest.mark.parametrize('T,K', [(1, 51200), (15, 51200), (63, 700), (64, 51200), (65, 51200),
                                 (255, 16), (256, 13), (257, 16), (1023, 3), (1024, 4), (1025, 4)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.float64])
def test_moments(T, K, dtype):
  """FP64 sums of T terms: within some 1e-13 of the terms."""
  g = torch.Generator(device='cuda').manual_seed(T)
  x = (3.0 + torch.randn(T, K, generator=g, device='cuda', dtype=torch.float64)).to(dtype)
  mean, var = readout.empirical_moments(x)
  r = x.double().cpu().numpy()
  np.testing.assert_allclose(mean.cpu().numpy().reshape(-1), r.mean(0), rtol=1e-13)
  np.testing.assert_allclose(var.cpu().numpy().reshape(-1), r.var(0), rtol=1e-12, atol=1e-26)


def test_few_rows_of_many_columns():
  """64 rows of 51,200 columns (13 MB) take no longer than the calls, as 64 of
  6000 do; in workgroups of 1024 threads three times as long."""
  from edward_amd import _lib as L
  from edward_amd.engine import Context
  ctx = Context()
  best = []
  for K in (6000, 51200):
    x = torch.randn(64, K, device='cuda')
    out = torch.empty(2, K, dtype=torch.float64, device='cuda')
    times = []
    for _ in range(20):
      a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      a.record()
      for _ in range(20):
        ctx.lib.edhmc_sample_moments(ctx.h, L.ptr(x), L.F32, 64, K, 0, L.ptr(out[0]),
                                     L.ptr(out[1]), ctx.stream)
      b.record()
      b.synchronize()
      times.append(a.elapsed_time(b))
    best.append(min(times))
  print('times', best, flush=True)
  assert best[1] < 1.8 * best[0], best
