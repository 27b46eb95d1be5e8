"""Autocovariances at all lags by transforms and the effective sample sizes
from them, at the edges of the transforms' lengths, against FP64 numpy."""

import numpy as np
import pytest
import torch

from edward_amd import diagnostics as dg

pytestmark = pytest.mark.gpu

# draws around the powers of two where the length doubles (and 2048, the last
# that takes transforms); odd numbers of chains; coordinates fewer and more
# than transforms side by side in a workgroup
SHAPES = [(4, 3, 2), (33, 1, 3), (64, 7, 1), (65, 2, 5), (128, 33, 2), (129, 4, 17), (257, 3, 33),
          (512, 5, 1), (513, 1, 2), (1000, 9, 64), (1024, 2, 3), (1025, 3, 2), (2048, 3, 2),
          (2049, 2, 2)]


def _store(T, C, D, seed=3):
  rng = np.random.default_rng(seed)
  x = rng.normal(size=(T, C, D))
  for t in range(1, T):
    x[t] += 0.8 * x[t - 1]
  return (x + 0.5 * rng.normal(size=(1, C, D)) + 10.0 * rng.normal(size=D)).astype(np.float32)


def _acov(x):
  a = x.astype(np.float64)
  a -= a.mean(0)
  T = len(a)
  return np.stack([(a[:T - l] * a[l:]).sum((0, 1)) / T for l in range(T)])


@pytest.mark.parametrize('T,C,D', SHAPES)
def test_all_lags(T, C, D):
  """Rounding of a transform is some log2(N) roundings (2^-53) of the root
  mean square: every lag within 1e-13 of the lag-0 sum."""
  from edward_amd.engine import Context
  x = _store(T, C, D)
  acov, cmean = dg.autocov(Context(), torch.as_tensor(x, device='cuda'), T - 1)
  ref = _acov(x)
  np.testing.assert_allclose(cmean.cpu().numpy(), x.astype(np.float64).mean(0), rtol=1e-12,
                             atol=1e-13 * np.abs(x).max())
  assert (np.abs(acov.cpu().numpy() - ref) <= 1e-13 * ref[0]).all()


@pytest.mark.parametrize('between', [True, False])
@pytest.mark.parametrize('T,C,D', SHAPES)
def test_ess(T, C, D, between):
  """The device's sum against the host's on the same definition: with every
  rho_t within 1e-13 the time tau, at most T of them, is within 2 T 1e-13 of
  its value times what it is at least (the floor is above 0.1)."""
  from edward_amd.engine import Context
  x = _store(T, C, D, 5)
  x[:, :, 0] = x[0, :, :1].T.reshape(C) if D > 1 else x[:, :, 0]   # a coordinate that never moves
  got = dg.ess(Context(), torch.as_tensor(x, device='cuda'), between=between)
  ref = dg.ess_from_acov(_acov(x), x.astype(np.float64).mean(0), T, between)
  np.testing.assert_allclose(got, ref, rtol=max(1e-10, 20 * T * 1e-13))


def test_not_finite():
  """A coordinate with an infinite draw has no effective samples; the others
  are untouched."""
  from edward_amd.engine import Context
  x = _store(300, 5, 4)
  ref = dg.ess(Context(), torch.as_tensor(x, device='cuda'))
  x[17, 2, 1] = np.inf
  got = dg.ess(Context(), torch.as_tensor(x, device='cuda'))
  assert got[1] == 0.0
  assert np.array_equal(np.delete(got, 1), np.delete(ref, 1))
