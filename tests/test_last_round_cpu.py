"""The items of a persistent position-wise pass (last_round, tile_piece in openfold-3_amd/csrc/of3_tiles.h) on the host:
every position of every tile belongs to exactly one item, and a launch with pieces ends with one round of them."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include "of3_tiles.h"
#include <cstdio>
#include <vector>
using namespace of3;
template <int PART> static bool covers(const LastRound& r, long tiles) {
  std::vector<char> seen(tiles * 128, 0);
  for (int item = 0; item < r.items; ++item) {
    const TilePiece p = tile_piece<PART>(item, r.whole);
    if (p.tile < 0 || p.tile >= tiles || p.first < 0 || p.first + p.count > 128 || p.count != 8 << p.group_bits) return false;
    if ((item < r.whole) != (p.count == 128)) return false;
    for (int k = 0; k < p.count; ++k) if (seen[p.tile * 128 + p.first + k]++) return false;
  }
  for (char c : seen) if (!c) return false;
  return true;
}
int main() {
  const int grids[] = {1, 2, 3, 8, 255, 256, 512};
  for (int grid : grids)
    for (long tiles = 1; tiles < 4L * grid + 3; ++tiles) {
      const LastRound r = last_round(tiles, grid);
      bool ok = r.piece == 128 ? covers<128>(r, tiles) : r.piece == 64 ? covers<64>(r, tiles) : r.piece == 32 && covers<32>(r, tiles);
      if (r.piece < 128) ok = ok && r.whole % grid == 0 && r.items - r.whole <= grid;
      else ok = ok && r.whole == r.items;
      if (!ok) return printf("grid %d tiles %ld piece %d\n", grid, tiles, r.piece), 1;
    }
  const LastRound half = last_round(256 + 94, 256), quarter = last_round(40, 256), none = last_round(256 + 200, 256);
  return half.piece == 64 && quarter.piece == 32 && none.piece == 128 ? 0 : 2;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_items_cover_every_position_once(tmp_path):
    src, exe = str(tmp_path / "check.cpp"), str(tmp_path / "check")
    with open(src, "w") as fh:
        fh.write(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "openfold-3_amd", "csrc"), src, "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
