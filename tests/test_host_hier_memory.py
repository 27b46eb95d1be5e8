"""Host side of the hierarchical model: the memory its gradient pass needs
beside the residuals."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')


@pytest.mark.parametrize('N,C', [(2000000, 256), (500000, 50)])
def test_fits_beside_the_residuals(N, C):
  """Residuals of C padded chains, twice X, and little else: where eta of all
  rows and chains does not fit beside them the form of the pass that keeps
  less of it runs (the residual-sized eta would be 2 GB here)."""
  host_calls.run('N, C = %d, %d\n' % (N, C) + r'''
G, D, MB = 100, 64, 1 << 20
off = (c.c_int64 * (G + 1))(*[N // G * g for g in range(G + 1)])
assert lib.edhmc_bind_hier(h, X, Y, off, G, N, D, None) == 0
assert lib.edhmc_hier_set_state(h, X, C, None) == 0
usual = kernels(log())
assert any('grad_rows_kernel' in k for k in usual)
residuals, eta = 256 * N * 4, C * N * 4
room = fake.fake_in_use() - eta + 64 * MB
h2 = h
lib.edhmc_destroy(h)
h = c.c_void_p()
assert lib.edhmc_create(0, c.byref(h)) == 0
fake.fake_limit(room)
assert lib.edhmc_bind_hier(h, X, Y, off, G, N, D, None) == 0
log()
assert lib.edhmc_hier_set_state(h, X, C, None) == 0, err()
tight = kernels(log())
assert any('grad_wide_kernel' in k for k in tight) and not any('grad_rows_kernel' in k for k in tight)
assert lib.edhmc_hier_transition(h, 0.1, 2, None, None, 1, 0, None, None, None, None) == 0
assert not any('grad_rows_kernel' in k for k in kernels(log()))
''')
