"""Host side of the readout calls: their scratch belongs to the context, so
calls on several streams take turns with it, and a captured call goes without."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')

_CALLS = r'''
CALLS = {
    'autocov_direct': lambda st: lib.edhmc_autocov(h, X, 500, 8, 10, 20, A, B, st),
    'autocov_means': lambda st: lib.edhmc_autocov(h, X, 500, 8, 10, 20, A, None, st),
    'autocov_all': lambda st: lib.edhmc_autocov(h, X, 500, 8, 10, 499, A, None, st),
    'autocov_long': lambda st: lib.edhmc_autocov(h, X, 5000, 8, 10, 64, A, B, st),
    'lags': lambda st: lib.edhmc_autocov_lags(h, X, 5000, 8, 10, 65, 66, B, A, st),
    'ess': lambda st: lib.edhmc_ess(h, X, 500, 8, 10, 1, A, st),
    'ess_short': lambda st: lib.edhmc_ess(h, X, 12, 8, 10, 1, A, st),
}
'''


def test_streams_take_turns():
  """Between the last kernel of a call and the first one of a call on another
  stream lie an event recorded on the one and waited for on the other."""
  host_calls.run(_CALLS + r'''
s1, s2 = p(11), p(12)
for n1, f1 in CALLS.items():
  for n2, f2 in CALLS.items():
    log()
    assert f1(s1) == 0, err()
    first = log()
    assert f2(s2) == 0, err()
    second = log()
    last = max(i for i, l in enumerate(first) if l[0] == 'launch')
    events = {l[2] for i, l in enumerate(first) if l[0] == 'record' and l[1] == '11' and i > last}
    start = min(i for i, l in enumerate(second) if l[0] == 'launch')
    waited = {l[2] for l in second[:start] if l[0] == 'wait' and l[1] == '12'}
    assert events & waited, (n1, n2, first, second)
''')


def test_captured_calls_use_no_scratch():
  """Under capture the autocovariances are made without memory of the
  context's (nothing allocated or freed, no event), also where a call before
  has left some; the effective sample size is refused before any launch."""
  host_calls.run(_CALLS + r'''
st = p(11)
for warm in (False, True):
  if warm:
    for f in CALLS.values():
      assert f(p(12)) == 0
  fake.fake_capture(st, 1)
  for n, f in CALLS.items():
    log()
    rc = f(st)
    calls = log()
    if n.startswith('ess'):
      assert rc == L.EUNSUPPORTED and 'captur' in err() and not calls, (n, rc, calls)
      continue
    assert rc == 0, (n, err())
    assert kernels(calls) and {l[0] for l in calls} == {'launch'}, (n, calls)
    assert not any('acov_power' in k for k in kernels(calls))
  fake.fake_capture(st, 0)
''')


def test_without_memory_for_scratch():
  """Where the device has no memory left the autocovariances still are made,
  as they are under capture."""
  host_calls.run(_CALLS + r'''
fake.fake_limit(fake.fake_in_use())
for n, f in CALLS.items():
  log()
  rc = f(p(11))
  if n.startswith('ess'):
    assert rc == L.ENOMEM, (n, rc)
  else:
    assert rc == 0 and any('autocov' in k for k in kernels(log())), (n, rc, err())
''')
