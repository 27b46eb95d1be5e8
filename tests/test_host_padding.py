"""Padding of the data rows, whatever tile shapes the library is built with."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which('hipcc') or '/opt/rocm/bin/hipcc'


@pytest.mark.skipif(not os.path.exists(HIPCC), reason='no hipcc')
@pytest.mark.parametrize('flags', [[], ['-DEDHMC_CFG_P2=1,2,2,2,64']])
def test_rows_fill_the_few_chain_tiles(tmp_path, flags):
  """The few-chain kernel reads whole tiles of X and y up to the padded rows:
  N_pad has to be a multiple of its longest tile, also with the narrower tiles
  that the forward pass may be built with."""
  src = tmp_path / 'padding.hip'
  src.write_text('#include "edhmc_glm.hip"\n'
                 'constexpr int longest = 16 * few_rb(16) * kFewWaves;\n'
                 'static_assert(longest == 256 && few_rb(32) <= few_rb(16) &&\n'
                 '              few_rb(256) <= few_rb(16), "longest tile");\n'
                 'static_assert(kRowPad % longest == 0, "row padding");\n')
  r = subprocess.run([HIPCC, '--offload-arch=gfx950', '--cuda-host-only', '-std=c++17',
                      '-fsyntax-only', '-I', os.path.join(ROOT, 'edward_amd', 'csrc')] + flags +
                     [str(src)], capture_output=True, text=True, timeout=300)
  assert r.returncode == 0, r.stderr[-2000:]
