"""Readout calls on two streams of one context, under capture and without
scratch, against calls made one at a time."""

import ctypes

import numpy as np
import pytest
import torch

from edward_amd import _lib as L
from edward_amd import diagnostics as dg

pytestmark = pytest.mark.gpu


def _store(T, C, D, seed):
  g = torch.Generator(device='cuda').manual_seed(seed)
  s = torch.randn(T, C, D, generator=g, device='cuda')
  for t in range(1, T):
    s[t] += 0.7 * s[t - 1]
  return s + torch.randn(D, generator=g, device='cuda')


# draws: transforms, direct sums; chains and coordinates that leave one group,
# several groups, narrow stores side by side
@pytest.mark.parametrize('shape,lag', [((1000, 256, 64), 999), ((1000, 64, 200), 20),
                                       ((2100, 100, 7), 64), ((300, 9, 300), 299)])
def test_two_streams(shape, lag):
  """Calls enqueued on two streams without waiting in between have the bits
  of calls made one after the other."""
  from edward_amd.engine import Context
  print('case', shape, lag, flush=True)
  eng = Context()
  a, b = _store(*shape, 1), _store(*shape, 2)
  ref = [dg.autocov(eng, x, lag) for x in (a, b)]
  torch.cuda.synchronize()
  streams = [torch.cuda.Stream(), torch.cuda.Stream()]
  for _ in range(3):
    out = []
    for k in range(6):
      with torch.cuda.stream(streams[k & 1]):
        out.append(dg.autocov(eng, (a, b)[k & 1], lag))
    torch.cuda.synchronize()
    for k, o in enumerate(out):
      assert torch.equal(o[0], ref[k & 1][0]) and torch.equal(o[1], ref[k & 1][1]), k


@pytest.mark.parametrize('means', [True, False])
@pytest.mark.parametrize('T,C,D,lag', [(200, 33, 5, 199), (500, 3, 130, 31), (2050, 2, 64, 70)])
def test_captured(T, C, D, lag, means):
  """A captured call makes its sums without scratch: its replays agree with
  the eager call to the rounding of the sums, some 1e-13 of lag 0's, whatever
  the context's own calls do in between."""
  from edward_amd.engine import Context
  print('case T=%d C=%d D=%d lag=%d %s' % (T, C, D, lag, means), flush=True)
  eng = Context()
  s = _store(T, C, D, 3)
  ref, mref = dg.autocov(eng, s, lag)
  other = _store(T + 1, C, D, 4)
  acov = torch.zeros_like(ref)
  cm = torch.zeros_like(mref)
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  with torch.cuda.graph(graph):
    eng.check(eng.lib.edhmc_autocov(eng.h, L.ptr(s), T, C, D, lag, L.ptr(acov),
                                    L.ptr(cm) if means else None, eng.stream))
    rc = eng.lib.edhmc_ess(eng.h, L.ptr(s), T, C, D, 1, L.ptr(acov), eng.stream)
  assert rc == L.EUNSUPPORTED
  for _ in range(3):
    acov.zero_()
    dg.autocov(eng, other, lag)
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    assert ((acov - ref).abs() <= 1e-13 * ref[0]).all()
    if means:
      assert torch.equal(cm, mref) or (cm - mref).abs().max() < 1e-13 * mref.abs().max()
