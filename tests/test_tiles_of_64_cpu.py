"""Tiles of 64 positions (openfold-3_amd/csrc/of3_tiles.h) on the host: rows, flat index space and the pieces of a last round cover every position
exactly once, in the ways the kernels walk them."""
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
constexpr int TP = 64;
static int rows(int N) {
  const RaggedTiles t = ragged_tiles<TP>(N);
  std::vector<int> cover(N * N, 0);
  const int Np = (N + 127) / 128 * 128;
  for (int tile = 0; tile < t.per_batch; ++tile) {
    const TilePlace p = N % TP ? tile_place<true, TP>(tile, N, t.full_per_row, t.tail_shift, t.per_batch, false)
                               : tile_place<false, TP>(tile, N, t.full_per_row, t.tail_shift, t.per_batch, false);
    if (p.i0 >= N || p.shift < 3 || p.shift > 6) return 1;
    for (int pos = 0; pos < TP; ++pos) {
      const int i = p.i0 + (pos >> p.shift), j = p.j0 + (pos & ((1 << p.shift) - 1));
      if (j >= Np) return 2;
      if (i < N && j < N) ++cover[i * N + j];
    }
  }
  for (int c : cover) if (c != 1) return 3;
  return 0;
}
static int flat(int N, int B) {
  const long long total = (long long)B * N * N;
  for (int tile = 0; tile * (long long)TP < total; ++tile) {
    const FlatTile t = flat_tile<TP>(tile, N, N * N, 1);  // the transposed view
    for (int d = 0; d < TP && tile * (long long)TP + d < total; ++d) {
      const long long p = tile * (long long)TP + d, b = p / (N * N), i = p / N % N, j = p % N;
      const long long got = N % TP == 0 ? flat_offset<0>(t, d, N, N * N, 1, N) : N >= TP ? flat_offset<1>(t, d, N, N * N, 1, N) : flat_offset<2>(t, d, N, N * N, 1, N);
      if (got != b * N * N + i + j * N) return 4;
    }
  }
  return 0;
}
static int items(long tiles, int grid) {
  const LastRound r = last_round<TP>(tiles, grid);
  std::vector<char> seen(tiles * TP, 0);
  if (r.piece != TP && (r.piece != 32 || r.whole % grid || r.items - r.whole > grid)) return 5;
  for (int item = 0; item < r.items; ++item) {
    const TilePiece p = r.piece == TP ? tile_piece<TP, TP>(item, r.whole) : tile_piece<32, TP>(item, r.whole);
    if (p.first + p.count > TP || p.count != 8 << p.group_bits) return 6;
    for (int k = 0; k < p.count; ++k) if (seen[p.tile * TP + p.first + k]++) return 7;
  }
  for (char c : seen) if (!c) return 8;
  return 0;
}
int main() {
  for (int N : {1, 7, 40, 63, 64, 65, 72, 96, 97, 104, 127, 128, 129, 161, 192, 200, 225, 300, 321})
    if (const int e = rows(N) + 10 * flat(N, 1) + 100 * flat(N, 3)) return printf("N %d: %d\n", N, e), 1;
  for (int grid : {1, 2, 7, 512, 768})
    for (long tiles = 1; tiles < 4L * grid + 3; ++tiles)
      if (const int e = items(tiles, grid)) return printf("grid %d, %ld tiles: %d\n", grid, tiles, e), 1;
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_every_position_once(tmp_path):
    src, exe = str(tmp_path / "check.cpp"), str(tmp_path / "check")
    with open(src, "w") as fh:
        fh.write(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I" + os.path.join(ROOT, "openfold-3_amd", "csrc"), src, "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
