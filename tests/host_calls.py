"""Runs calls of libedhmc.so on a HIP runtime without a device
(``fake_hip.cpp``), in a process of its own: what the host side allocates,
launches and waits for."""

import os
import subprocess
import sys
import tempfile

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, 'edward_amd', 'libedhmc.so')

_PRELUDE = r'''
import ctypes, importlib.util, sys, types
c = ctypes
fake = c.CDLL(%(fake)r, mode=c.RTLD_GLOBAL)
fake.fake_log.restype = c.c_char_p
fake.fake_in_use.restype = c.c_size_t
fake.fake_limit.argtypes = [c.c_size_t]
fake.fake_capture.argtypes = [c.c_void_p, c.c_int]
fake.fake_fail_kernel.argtypes = [c.c_char_p]
sys.modules['torch'] = types.ModuleType('torch')   # it would load the real runtime's users
spec = importlib.util.spec_from_file_location('_lib', %(binding)r)
L = importlib.util.module_from_spec(spec)
spec.loader.exec_module(L)
lib = L.load(%(lib)r)
p = lambda n: c.c_void_p(n)      # a device address that nothing reads
X, Y, A, B = p(1 << 40), p(2 << 40), p(3 << 40), p(4 << 40)
h = c.c_void_p()
assert lib.edhmc_create(0, c.byref(h)) == 0

def err():
  return lib.edhmc_last_error(h).decode()

def log():
  """The calls since the last log(): lists of words."""
  out = [l.split(' ') for l in fake.fake_log().decode().splitlines()]
  fake.fake_clear()
  return out

def kernels(calls):
  return [l[3] for l in calls if l[0] == 'launch']

log()
'''

_built = None


def _fake():
  global _built
  if _built is None:
    d = tempfile.mkdtemp(prefix='fake_hip_')
    _built = os.path.join(d, 'fake_hip.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', '-o', _built,
                    os.path.join(ROOT, 'tests', 'fake_hip.cpp')], check=True)
  return _built


def run(body):
  """Runs ``body`` after the prelude above; fails with what it printed."""
  code = _PRELUDE % dict(fake=_fake(), lib=LIB,
                         binding=os.path.join(ROOT, 'edward_amd', '_lib.py')) + body
  r = subprocess.run([sys.executable, '-c', code], capture_output=True, text=True, timeout=120)
  assert r.returncode == 0, r.stdout + r.stderr
