"""Host side of binding data: what it launches."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')


def test_launches():
  """One launch for the layouts of X, one each for y and the two prior
  vectors, whichever copies the compute type and width ask for: a minibatch is
  bound every update."""
  host_calls.run(r'''
for D, dtype in ((10, 0), (100, 0), (256, 0), (300, 0), (100, 1)):
  log()
  assert lib.edhmc_bind_glm(h, X, L.F32, Y, 1000, D, 0, 1.0, A, B, dtype, None) == 0, err()
  names = kernels(log())
  assert len(names) == 4 and sum('pad_copy' in n for n in names) == 3, (D, dtype, names)
''')
