"""The order in which workgroups take the tiles of a launch (decode_block, first_of_two), compiled for the host: every tile of every slice
is handed out exactly once, whatever the numbers of tiles and slices, the tiles of an XCD come heaviest first where that is asked for, and under a mask
no XCD has more work than the others."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
_PROGRAM = r"""
#include <cstdio>
#include <set>
#include <utility>
#include "fhog_bf16_util.h"
using namespace fhog::bf16k;
int main() {
  const int tiles[] = {1, 2, 3, 4, 5, 7, 8, 13, 16, 31, 32, 33, 63, 64, 65, 130}, slices[] = {1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 25, 36, 63, 64, 100};
  for (int T : tiles) for (int B : slices) for (int mode = 0; mode < 8; mode++) {
    const bool major = mode & 1, pairs = mode & 2, two = mode & 4;
    const unsigned grid = grid_blocks(T, B);
    std::set<std::pair<int, int>> seen[2];
    int last_tile[8] = {};
    for (unsigned i = 0; i < (two ? 2 * grid : grid); i++) {
      int id = (int)i, bh, tile;
      const int side = two && !first_of_two((int)grid, (int)grid, mode & 1, pairs, id);
      if (!decode_block(T, B, false, major, bh, tile, pairs && !two, id)) continue;
      if (bh < 0 || bh >= B || tile < 0 || tile >= T || !seen[side].insert({bh, tile}).second) return printf("%d tiles, %d slices, mode %d, id %u\n", T, B, mode, i), 1;
      // tile by tile: nothing follows lighter tiles of the XCD's own slices
      if (major && !pairs && !two && tile < last_tile[i % 8]) return printf("order: %d tiles, %d slices, id %u\n", T, B, i), 1;
      if (bh < B / 8 * 8) last_tile[i % 8] = tile;
    }
    for (int side = 0; side <= (two ? 1 : 0); side++)
      if ((int)seen[side].size() != T * B) return printf("%d tiles, %d slices, mode %d: %zu\n", T, B, mode, seen[side].size()), 1;
  }
  return 0;
}
"""


# the work of a tile grows with its index; slices in tile-major order and one after the other. Whole slices weigh the same on every XCD;
# the dealt ones are taken by turns, which leaves two of the heaviest tiles between the XCDs at most
_BALANCE = r"""
#include <cstdio>
#include "fhog_bf16_util.h"
using namespace fhog::bf16k;
int main() {
  const int tiles[] = {8, 31, 64, 128, 143, 300};
  for (int T : tiles) for (int B = 1; B <= 20; B++) for (int mode = 0; mode < 4; mode++) {
    long work[8] = {}, lo = 1L << 60, hi = 0;
    int count = 0;
    for (unsigned i = 0; i < grid_blocks(T, B); i++) {
      int bh, tile;
      if (!decode_block<MASK_CAUSAL>(T, B, mode & 2, mode & 1, bh, tile, false, (int)i)) continue;
      if (bh < 0 || bh >= B || tile < 0 || tile >= T) return printf("range: %d tiles, %d slices, mode %d, id %u\n", T, B, mode, i), 1;
      work[i & 7] += tile + 1, count++;
    }
    for (long w : work) lo = w < lo ? w : lo, hi = w > hi ? w : hi;
    if (count != T * B || hi - lo > 2 * T) return printf("%d tiles, %d slices, mode %d: %d tiles, work %ld to %ld\n", T, B, mode, count, lo, hi), 1;
  }
  return 0;
}
"""

# two sweeps of unequal length in one launch, tile by tile in turn: every tile of both exactly once, and at turn k neither is ahead of the other
_TURNS = r"""
#include <cstdio>
#include <set>
#include <utility>
#include "fhog_bf16_util.h"
using namespace fhog::bf16k;
int main() {
  const int tiles[] = {1, 2, 5, 8, 13, 31, 64, 65, 130};
  for (int TQ : tiles) for (int TK : tiles) for (int B = 1; B <= 12; B++) for (int pairs = 0; pairs < 2; pairs++) {
    const int gq = grid_blocks(TQ, B), gk = grid_blocks(TK, B);
    std::set<std::pair<int, int>> seen[2];
    int turns[8][2] = {};
    for (int i = 0; i < gq + gk; i++) {
      int id = i, bh, tile;
      const int side = !first_of_two(gq, gk, true, pairs, id), T = side ? TK : TQ;
      if (id < 0 || id >= (side ? gk : gq)) return printf("id: %d and %d tiles, %d slices, id %d\n", TQ, TK, B, i), 1;
      if (!pairs && (i >> 3) < 2 * (gq < gk ? gq : gk) / 8) {
        turns[i & 7][side]++;
        if (turns[i & 7][0] - turns[i & 7][1] < 0 || turns[i & 7][0] - turns[i & 7][1] > 1) return printf("turns: %d and %d tiles, %d slices, id %d\n", TQ, TK, B, i), 1;
      }
      if (!decode_block<MASK_CAUSAL>(T, B, !side, true, bh, tile, false, id)) continue;
      if (bh < 0 || bh >= B || tile < 0 || tile >= T || !seen[side].insert({bh, tile}).second) return printf("%d and %d tiles, %d slices, id %d\n", TQ, TK, B, i), 1;
    }
    if ((int)seen[0].size() != TQ * B || (int)seen[1].size() != TK * B) return printf("%d and %d tiles, %d slices\n", TQ, TK, B), 1;
  }
  return 0;
}
"""


def _run(tmp_path, program):
    src = tmp_path / "order.hip"
    src.write_text(program)
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = tmp_path / "order"
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", f"-I{ROOT}/include", f"-I{ROOT}/flash-hob_amd/csrc", str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout


_needs_hipcc = pytest.mark.skipif(not shutil.which("hipcc") and not Path("/opt/rocm/bin/hipcc").exists(), reason="needs hipcc")


@_needs_hipcc
def test_every_tile_once(tmp_path):
    _run(tmp_path, _PROGRAM)


@_needs_hipcc
def test_xcds_have_the_same_work_under_a_mask(tmp_path):
    _run(tmp_path, _BALANCE)


@_needs_hipcc
def test_sweeps_of_unequal_length_take_turns(tmp_path):
    _run(tmp_path, _TURNS)
