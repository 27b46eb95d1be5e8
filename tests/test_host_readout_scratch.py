"""Host side of the readout calls: the scratch the context keeps is bounded
whatever the width of the store."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')


# draws on both sides of each length of the transforms and of the last that
# takes them; coordinates from one to a hierarchical model of 100,000 groups
@pytest.mark.parametrize('D', [1, 33, 2048, 2049, 4097, 100000])
@pytest.mark.parametrize('T', [12, 64, 65, 1000, 1025, 2048, 2049])
def test_bounded(T, D):
  host_calls.run('T, D = %d, %d\n' % (T, D) + r'''
MB = 1 << 20
for C in (1, 2, 7, 300):
  h = c.c_void_p()
  assert lib.edhmc_create(0, c.byref(h)) == 0
  base = fake.fake_in_use()
  assert lib.edhmc_autocov(h, X, T, C, D, min(64, T - 1), A, B, None) == 0
  assert lib.edhmc_autocov(h, X, T, C, D, T - 1, A, B, None) == 0
  assert lib.edhmc_autocov_lags(h, X, T, C, D, 3, T - 3, B, A, None) == 0
  got = fake.fake_in_use() - base
  assert got <= (256 + 128) * MB, (C, got / MB)
  assert lib.edhmc_ess(h, X, T, C, D, 1, A, None) == 0
  got = fake.fake_in_use() - base
  mean = C * D * 8 + 16 * D              # chain means, their moments
  lags = T * D * 8 if T > 2048 else 32 * MB
  assert got <= (256 + 128) * MB + mean + lags, (C, got / MB)
  lib.edhmc_destroy(h)
  assert fake.fake_in_use() == base
''')


def test_lags_of_many_draws():
  """A narrow store's lags in windows of at most 128 MB of partial sums."""
  host_calls.run(r'''
base = fake.fake_in_use()
assert lib.edhmc_autocov(h, X, 1000000, 40, 1, 999999, A, B, None) == 0
assert fake.fake_in_use() - base <= 128 << 20, fake.fake_in_use() - base
calls = [l for l in log() if l[0] == 'launch' and 'autocov_kernel' in l[3]]
assert len(calls) > 1
''')
