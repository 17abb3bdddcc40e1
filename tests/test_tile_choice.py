"""The GEMMs' tile models (csrc/tile_choice.h), compiled for the host: no choice is
much slower than the fastest kernel measured for the shape."""
from __future__ import annotations

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <stdio.h>
#include <stdlib.h>
#include "tile_choice.h"
using namespace ipus;
int main(int argc, char** argv) {
  for (int i = 2; i + 4 < argc; i += 5) {
    auto n = [&](int k) { return (uint32_t)strtoul(argv[i + k], nullptr, 10); };
    if (argv[1][0] == '1')
      printf("%u\n", gemm_f16_tile(n(0), n(1), n(2), n(3), (GemmAccess)n(4)));
    else
      printf("%d\n", (int)tile_f32(n(0), n(1), n(2), n(3), n(4) != 0));
  }
}
"""

CHUNK, DWORD, ELEMENT = 0, 1, 2
# (M, N, K, batches, access): kernel us by tile.
F16 = {
    (4096, 4096, 8, 1, CHUNK): {256: 10.1, 128: 18.3, 64: 22.8, 32: 60.7},
    (4096, 4096, 256, 1, CHUNK): {256: 14.7, 128: 22.2, 64: 28.8, 32: 69.8},
    (4096, 4096, 2048, 1, CHUNK): {256: 51.9, 128: 66.3, 64: 96.6, 32: 230.8},
    (8192, 8192, 64, 1, CHUNK): {256: 42.8, 128: 60.9, 64: 82.6, 32: 244.4},
    (3072, 3072, 64, 1, CHUNK): {256: 8.2, 128: 13.0, 64: 14.0, 32: 35.6},
    (3072, 3072, 640, 1, CHUNK): {256: 17.6, 128: 22.5, 64: 24.7, 32: 55.5},
    (2592, 4368, 440, 1, CHUNK): {256: 18.6, 128: 22.8, 64: 29.3, 32: 66.2},
    (3093, 1976, 64, 1, CHUNK): {256: 8.3, 128: 9.2, 64: 9.6, 32: 24.7},
    (3093, 1976, 1024, 1, CHUNK): {256: 23.2, 128: 21.0, 64: 26.0, 32: 59.2},
    (2048, 2048, 64, 1, CHUNK): {256: 7.9, 128: 5.9, 64: 7.5, 32: 16.8},
    (2048, 2048, 2048, 1, CHUNK): {256: 37.4, 128: 18.4, 64: 26.9, 32: 59.8},
    (4952, 224, 40, 1, CHUNK): {256: 8.1, 128: 5.4, 64: 4.6, 32: 7.0},
    (4952, 224, 2048, 1, CHUNK): {256: 36.0, 128: 16.0, 64: 15.9, 32: 19.2},
    (1024, 1024, 64, 1, CHUNK): {256: 7.3, 128: 5.1, 64: 3.4, 32: 5.7},
    (1024, 1024, 2048, 1, CHUNK): {256: 35.5, 128: 15.4, 64: 7.8, 32: 15.9},
    (729, 1152, 128, 1, CHUNK): {256: 8.4, 128: 5.5, 64: 3.6, 32: 5.7},
    (729, 4304, 1024, 1, CHUNK): {256: 23.3, 128: 11.0, 64: 17.2, 32: 31.4},
    (16, 4096, 256, 1, CHUNK): {256: 9.0, 128: 5.4, 64: 3.6, 32: 2.9},
    (256, 256, 256, 1, CHUNK): {256: 9.0, 128: 5.5, 64: 3.5, 32: 3.1},
    (64, 64, 2048, 1, CHUNK): {256: 34.9, 128: 13.0, 64: 6.7, 32: 4.7},
    (512, 512, 8, 12, CHUNK): {256: 7.8, 128: 5.9, 64: 6.7, 32: 13.2},
    (100, 64, 256, 300, DWORD): {256: 21.4, 128: 10.5, 64: 7.6, 32: 16.9},
    (1500, 1500, 64, 1, DWORD): {256: 11.0, 128: 6.0, 64: 6.5, 32: 10.6},
    (112, 1190, 184, 36, DWORD): {256: 14.7, 128: 11.4, 64: 10.5, 32: 23.4},
    (4095, 4097, 65, 1, ELEMENT): {128: 26.4, 64: 27.2, 32: 71.6},
    (4095, 4097, 441, 1, ELEMENT): {128: 50.8, 64: 56.6, 32: 167.7},
    (1023, 1025, 13, 1, ELEMENT): {128: 5.7, 64: 4.4, 32: 7.6},
    (1023, 1025, 441, 1, ELEMENT): {128: 10.2, 64: 7.9, 32: 15.5},
    (255, 257, 251, 1, ELEMENT): {128: 7.6, 64: 5.6, 32: 4.3},
}
# (M, N, K, batches, whole 16-byte chunks): kernel us on 128 x 128, 64 x 64 and 32 x
# 32 tiles (128 x 128 only where the operands are whole chunks).
F32 = {
    (4096, 4096, 8, 1, 1): (21.0, 31.8, 67.6), (4096, 4096, 64, 1, 1): (29.2, 38.3, 63.0),
    (4096, 4096, 1000, 1, 1): (273.8, 272.6, 330.2), (4096, 4096, 2, 1, 0): (48.1, 32.4, 78.8),
    (2392, 2688, 8, 1, 1): (12.2, 16.6, 29.5), (2392, 2688, 256, 1, 1): (42.7, 37.7, 46.5),
    (2760, 960, 64, 1, 1): (9.4, 8.8, 12.8), (1024, 1024, 8, 1, 1): (6.8, 4.2, 6.2),
    (1024, 1024, 1000, 1, 1): (76.0, 21.6, 24.1), (256, 256, 256, 1, 1): (21.0, 7.0, 4.0),
    (256, 256, 1000, 1, 1): (75.5, 19.5, 6.9), (8192, 64, 256, 1, 1): (21.5, 7.2, 5.9),
    (800, 1088, 8, 4, 1): (8.1, 9.3, 15.8), (3336, 298, 8, 8, 0): (33.8, 19.4, 39.7),
    (108, 384, 2, 26, 0): (11.1, 5.8, 8.2), (1960, 1400, 144, 17, 1): (152.3, 185.0, 262.9),
}


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no host compiler")
    tmp = tmp_path_factory.mktemp("choice")
    (tmp / "choice.cpp").write_text(SOURCE)
    subprocess.run([compiler, "-std=c++17", "-I", os.path.join(ROOT, "ipu-stack_amd", "csrc"),
                    "-o", str(tmp / "choice"), str(tmp / "choice.cpp")], check=True)

    def run(kind, shapes):
        out = subprocess.run([str(tmp / "choice"), kind] + [str(n) for s in shapes for n in s],
                             check=True, capture_output=True, text=True).stdout
        return [int(line) for line in out.split()]

    return run


def test_f16_tile_is_near_the_fastest(choose):
    for (shape, us), tile in zip(F16.items(), choose("16", F16)):
        # a small product's kernels differ by little more than the timing does
        assert us[tile] <= 1.1 * min(us.values()) + 0.3, (shape, tile)


def test_f16_tile_of_the_longest_rows(choose):
    """Counts of tiles past 32 bits, and no K at all (only the element form takes it)."""
    shapes = [(2 ** 31 - 1, 2 ** 31 - 1, 8, 1, CHUNK), (2 ** 31 - 1, 8, 8, 1, CHUNK), (8, 8, 0, 1, ELEMENT),
              (2 ** 31 - 1, 2 ** 20, 2 ** 20, 65535, ELEMENT)]
    assert choose("16", shapes) == [256, 64, 32, 128]


def test_f32_tile_is_near_the_fastest(choose):
    for (shape, us), kernel in zip(F32.items(), choose("32", F32)):
        assert shape[4] or kernel != 0, shape
        assert us[kernel] <= 1.1 * min(us) + 0.3, (shape, kernel)
