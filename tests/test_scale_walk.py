"""The walk over a row's scales of the direct-to-LDS GEMM (dq_scale_walk.h), on the host: nothing is read outside the array, and
every group lies where the kernel looks for it while its tile is multiplied."""

import os
import shutil
import subprocess

import pytest

from tilelang_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "dq_scale_walk.h"
#include <cstdio>
#include <cstring>
#include <vector>
using dq::gemm::ScaleWalk;

// tiles_per_stage: of 64 k; shift: log2(tiles of 64 k in a group); rows of `groups` groups
static int check(int rows, int groups, int shift, int tiles_per_stage) {
  const bool odd = groups & 1;
  std::vector<unsigned short> array(rows * groups);
  for (size_t i = 0; i < array.size(); ++i) array[i] = (unsigned short)(i + 1);
  const size_t size = 2 * array.size();
  const int stages = (groups << shift) / tiles_per_stage;
  for (int lane = 0; lane < (rows + 3 & ~1); ++lane) {  // lanes beyond the matrix hold its last row
    const int row = lane < rows ? lane : rows - 1;
    const ScaleWalk walk(row, groups, odd);
    const bool ahead = odd && (lane & 1);
    unsigned char ring[4096];
    std::memset(ring, 0xFF, sizeof ring);
    auto load = [&](size_t from, unsigned bytes, int slot) -> bool {
      if (from + bytes > size || from % 4 != 0) { std::printf("row %d of %d, %d groups: bytes %zu .. %zu of %zu\n", row, rows, groups, from, from + bytes, size); return false; }
      std::memset(ring + slot * 1024, 0, 4);
      std::memcpy(ring + slot * 1024, (const char*)array.data() + from, bytes);
      return true;
    };
    if (odd && !load(walk.start, 4, 3)) return 1;
    auto issue = [&](int stage) -> bool {  // with the first tile that a dword serves
      const int tile = stage * tiles_per_stage, dword = tile >> (shift + 1);
      if (tile & ((2 << shift) - 1)) return true;
      return load(walk.from(dword) + 4 * (size_t)dword, 4, dword & 3);
    };
    if (!issue(0) || (stages > 1 && !issue(1))) return 1;
    for (int stage = 0; stage < stages; ++stage) {
      if (stage + 2 < stages && !issue(stage + 2)) return 1;  // in flight while this one is multiplied
      for (int tile = stage * tiles_per_stage; tile < (stage + 1) * tiles_per_stage; ++tile) {
        const int group = tile >> shift;
        unsigned short got;
        std::memcpy(&got, ring + (ahead ? ScaleWalk::one_ahead(group) : ScaleWalk::aligned(group)), 2);
        if (lane == row && got != array[(size_t)row * groups + group]) { std::printf("row %d, group %d of %d\n", row, group, groups); return 1; }
      }
    }
  }
  return 0;
}

int main() {
  for (int rows = 1; rows <= 6; ++rows)  // (the choice of the kernel keeps an odd count of both away from it)
    for (int shift = 0; shift <= 3; ++shift)
      for (int groups = 2; groups <= 41; ++groups)
        for (int tiles_per_stage = 1; tiles_per_stage <= 2; ++tiles_per_stage)
          if (!(rows & groups & 1) && (groups << shift) % tiles_per_stage == 0 && check(rows, groups, shift, tiles_per_stage)) return 1;
  return 0;
}
"""


def test_every_load_lies_in_the_array_and_every_group_where_it_is_read(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    source, program = tmp_path / "walk.cpp", tmp_path / "walk"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "tilelang_amd", "csrc"), str(source), "-o", str(program)], check=True)
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=60)
    assert done.returncode == 0, done.stdout


@pytest.mark.parametrize("operands,K,group,mode", [(1, 1088, 0, 0), (0, 1088, 64, 3), (0, 1152, 128, 5), (0, 1792, 256, 5)])
def test_an_odd_count_of_groups_goes_with_an_even_count_of_rows(operands, K, group, mode):
    rows = _lib.load_library().dq_tile_rows
    assert rows(operands, 2570, 5131, K, group, mode) == 0 and rows(operands, 2570, 5132, K, group, mode) > 0
    assert rows(operands, 2570, 5131, 2 * K, group, mode) > 0
