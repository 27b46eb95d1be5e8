"""Engines that the garbage collector finds during a graph capture."""

import gc

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_collected_during_capture():
  """Freeing a context waits for the device and frees memory, neither of which
  a capture allows: one collected there is freed later, and the capture goes
  on."""
  from edward_amd import engine
  from edward_amd.engine import Context, GLMEngine
  x = torch.ones(1000, device='cuda')
  gc.collect()
  Context().close()
  eng = GLMEngine(np.ones((20, 3), np.float32), np.ones(20, np.float32))
  eng.set_state(np.zeros((2, 3), np.float32))
  eng.itself = eng            # a cycle: only the collector finds it
  del eng
  torch.cuda.synchronize()
  graph = torch.cuda.CUDAGraph()
  gc.disable()                # not before the capture
  try:
    with torch.cuda.graph(graph):
      gc.collect()
      y = x * 2.0
  finally:
    gc.enable()
  for _ in range(3):
    y.zero_()
    torch.cuda.synchronize()
    graph.replay()
    torch.cuda.synchronize()
    assert bool((y == 2.0).all())
  assert len(engine._deferred) == 1
  Context().close()
  assert not engine._deferred
