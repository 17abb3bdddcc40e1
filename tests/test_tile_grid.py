"""The GEMM tile kernels' grid (csrc/tile_grid.h), compiled for the host: within
HIP's limit of fewer than 2^32 work-items per dimension, every tile once."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "tile_grid.h"
using namespace ipus;
int main(int argc, char** argv) {
  for (int i = 1; i < argc; ++i) {
    const uint64_t tiles = strtoull(argv[i], nullptr, 10);
    const TileGrid g = tile_grid(tiles);
    // Tile ids run through 0 .. x z - 1 without a gap: the first and last of each z.
    bool whole = true;
    for (uint32_t z = 0; z < g.z; ++z)
      whole = whole && grid_tile(0, z) == (uint64_t)z * g.x && grid_tile(g.x - 1, z) == (uint64_t)(z + 1) * g.x - 1;
    printf("%u %u %d\n", g.x, g.z, whole);
  }
}
"""

TILES = [1, 7, 128, (1 << 22) - 1, 1 << 22, (1 << 22) + 1, 1 << 23, (1 << 24) - 3,
         (1 << 29) // 32, ((1 << 31) - 1 + 63) // 64, ((1 << 31) - 1 + 31) // 32, (1 << 31) - 1]


def test_grid_covers_every_tile_within_the_launch_limit(tmp_path):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host compiler")
    (tmp_path / "grid.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-I", os.path.join(ROOT, "ipu-stack_amd", "csrc"),
                    "-o", str(tmp_path / "grid"), str(tmp_path / "grid.cpp")], check=True)
    out = subprocess.run([str(tmp_path / "grid")] + [str(t) for t in TILES], check=True,
                         capture_output=True, text=True).stdout.split("\n")
    for tiles, line in zip(TILES, out):
        x, z, whole = map(int, line.split())
        assert whole and x * 512 < 1 << 32 and z <= 65535, tiles
        assert 0 <= x * z - tiles < x, tiles  # no tile left out, no z without one
        assert z == 1 or x % 8 == 0, tiles    # the XCD of a tile is its id modulo 8
