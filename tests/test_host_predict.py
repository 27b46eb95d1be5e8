"""Host side of the posterior predictive: what repeated calls allocate."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')


def test_repeated_calls_allocate_nothing():
  """With and without replicates in turn (other kernels, other partial sums),
  and without the mean: after one of each nothing is allocated or freed."""
  host_calls.run(r'''
for D, dtype in ((20, 0), (200, 0), (300, 0), (100, 1)):
  assert lib.edhmc_bind_glm(h, X, L.F32, Y, 5000, D, 0, 1.0, A, B, dtype, None) == 0
  for k in range(3):
    if k == 1:
      log()
    for mean, rep in ((A, None), (A, B), (None, None), (A, B), (A, None)):
      assert lib.edhmc_predict(h, X, 300, mean, Y, rep, 1, None) == 0, err()
  calls = log()
  assert not [l for l in calls if l[0] in ('malloc', 'free')], (D, dtype, calls[:40])
''')
