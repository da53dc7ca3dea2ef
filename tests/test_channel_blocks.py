"""The channel blocks of the transposes, to and from the cells' rows and of planar
features (``csrc/channel_blocks.h``), compiled
for the host: for every channel count the blocks lie inside the row, cover it,
are no wider than the LDS tile and hold at least one whole piece, which the
kernels' 16-byte accesses rely on."""
from __future__ import annotations

import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / 'bevfusion-triton_amd' / 'csrc'

PROGRAM = r'''
#include <cstdio>
#include <initializer_list>
#include "channel_blocks.h"
using namespace channel_blocks;

// blocks of `width` nominal channels of a row of C, moved in pieces
static int check(const char *what, int C, int width, int limit, int piece) {
  int covered = 0, last = 0;
  for (int cn = 0; cn < C; cn += width) {
    const int c0 = first_channel(C, piece, cn);
    const int cb = C - c0 < width ? C - c0 : width;
    if (c0 < 0 || c0 > covered || cb < piece || cb > limit || c0 + cb > C) last = 1;
    if (c0 + cb > covered) covered = c0 + cb;
  }
  if (last || covered != C || width < 1) {
    std::printf("%s: C=%d width=%d piece=%d\n", what, C, width, piece);
    return 1;
  }
  return 0;
}

int main() {
  int bad = 0;
  for (int C = 1; C <= 20000; ++C)
    for (int piece : {1, 4, 8})
      if (C >= piece)
        bad += check("tile_channels", C, tile_channels(C), kTileChannels, piece);
  for (int C = 4; C <= 20000; ++C) {
    bad += check("planar_channels", C, planar_channels(C), kPlanarChannels, 4);
    bad += planar_blocks(C) * planar_channels(C) < C ||
           (planar_blocks(C) - 1) * planar_channels(C) >= C;
  }
  return bad ? 1 : 0;
}
'''


def test_every_block_holds_a_piece(tmp_path):
    cxx = shutil.which('g++') or shutil.which('c++')
    if cxx is None:
        pytest.skip('no host C++ compiler')
    src, exe = tmp_path / 'blocks.cpp', tmp_path / 'blocks'
    src.write_text(PROGRAM)
    subprocess.run([cxx, '-std=c++17', '-O1', '-Wall', '-Werror', f'-I{CSRC}', str(src), '-o',
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
