"""Host side of the chain state's allocations: after one that fails, the same
call starts over instead of taking what is there for ready."""

import os

import pytest

import host_calls

pytestmark = pytest.mark.skipif(not os.path.exists(host_calls.LIB), reason='library not built')

# rows, columns, chains, compute type: few chains with and without a narrower
# copy of X, one pass over X in both forms, two products in both types
GLM = [(3000, 10, 2, 0), (3000, 64, 4, 0), (3000, 100, 50, 0), (70000, 60, 600, 0),
       (3000, 300, 2, 0), (3000, 100, 50, 1), (20000, 512, 300, 1)]


@pytest.mark.parametrize('N,D,C,dtype', GLM)
def test_set_state(N, D, C, dtype):
  """Whichever allocation of a set_state fails, it launches nothing after
  that, the chains are not ready, and the same call made again allocates what
  a first call does."""
  host_calls.run('N, D, C, dtype = %d, %d, %d, %d\n' % (N, D, C, dtype) + r'''
def fresh():
  global h
  h = c.c_void_p()
  assert lib.edhmc_create(0, c.byref(h)) == 0
  base = fake.fake_in_use()
  assert lib.edhmc_bind_glm(h, X, L.F32, Y, N, D, 0, 1.0, A, B, dtype, None) == 0
  log()
  return base

base = fresh()
assert lib.edhmc_set_state(h, X, C, None) == 0
whole, calls = fake.fake_in_use() - base, log()
lib.edhmc_destroy(h)
n = 1
while True:
  base = fresh()
  fake.fake_fail_malloc(n)
  rc = lib.edhmc_set_state(h, X, C, None)
  if fake.fake_to_fail():          # fewer allocations than that
    fake.fake_fail_malloc(0)
    assert rc == 0
    break
  failed = log()
  at = [l[0] for l in failed].index('malloc_failed')
  if rc == 0:      # eta's: the form that needs less of it
    assert any('grad_wide' in k for k in kernels(failed)), (n, failed)
    lib.edhmc_destroy(h)
    n += 1
    continue
  assert rc == L.ENOMEM and not kernels(failed[at:]), (n, rc, failed)
  assert lib.edhmc_run(h, 0.1, 2, X, 3, 0, 3, 1, 0, None, None) == L.ESTATE
  assert lib.edhmc_moments_enable(h, 1) == L.ESTATE
  log()
  assert lib.edhmc_set_state(h, X, C, None) == 0, (n, err())
  again = log()
  assert kernels(again) == kernels(calls), (n, again)
  assert fake.fake_in_use() - base == whole, (n, fake.fake_in_use() - base, whole)
  lib.edhmc_destroy(h)
  n += 1
assert n > 10, n
''')


def test_failed_copy_of_x():
  """The narrower copy of X is made again where its kernel did not launch."""
  host_calls.run(r'''
assert lib.edhmc_bind_glm(h, X, L.F32, Y, 3000, 10, 0, 1.0, A, B, 0, None) == 0
fake.fake_fail_kernel(b'few_layout')
assert lib.edhmc_set_state(h, X, 2, None) == L.EHIP
fake.fake_fail_kernel(b'')
log()
assert lib.edhmc_set_state(h, X, 2, None) == 0
assert any('few_layout' in k for k in kernels(log()))
''')


def test_hierarchical():
  """The same for the hierarchical model, whose data may fail to bind too."""
  host_calls.run(r'''
G, N, D, C = 40, 4000, 12, 70
off = (c.c_int64 * (G + 1))(*[100 * g for g in range(G + 1)])

def bind():
  return lib.edhmc_bind_hier(h, X, Y, off, G, N, D, None)

n = 1
while True:
  h = c.c_void_p()
  assert lib.edhmc_create(0, c.byref(h)) == 0
  fake.fake_fail_malloc(n)
  rc = bind()
  if fake.fake_to_fail():
    fake.fake_fail_malloc(0)
    break
  assert rc == L.ENOMEM, (n, rc)
  log()
  assert lib.edhmc_hier_set_state(h, X, C, None) == L.ESTATE, n
  assert lib.edhmc_set_state(h, X, C, None) == L.ESTATE, n
  assert not kernels(log())
  assert bind() == 0 and lib.edhmc_hier_set_state(h, X, C, None) == 0
  lib.edhmc_destroy(h)
  n += 1
assert n > 8, n

log()
base = fake.fake_in_use()
assert lib.edhmc_hier_set_state(h, X, C, None) == 0
whole, calls = fake.fake_in_use(), log()
n = 1
while True:
  assert bind() == 0
  assert lib.edhmc_hier_set_state(h, X, C + 300, None) == 0   # a state of other chains
  log()
  fake.fake_fail_malloc(n)
  rc = lib.edhmc_hier_set_state(h, X, C, None)
  if fake.fake_to_fail():
    fake.fake_fail_malloc(0)
    assert rc == 0
    break
  failed = log()
  at = [l[0] for l in failed].index('malloc_failed')
  if rc == 0:
    assert any('grad_wide' in k for k in kernels(failed)), (n, failed)
    n += 1
    continue
  assert rc == L.ENOMEM and not kernels(failed[at:]), (n, rc, failed)
  assert lib.edhmc_hier_transition(h, 0.1, 2, None, None, 1, 0, None, None, None, None) == L.ESTATE
  log()
  assert lib.edhmc_hier_set_state(h, X, C, None) == 0, (n, err())
  assert kernels(log()) == kernels(calls), n
  assert fake.fake_in_use() == whole, (n, fake.fake_in_use(), whole)
  n += 1
assert n > 15, n
''')
