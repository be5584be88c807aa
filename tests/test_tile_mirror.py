"""CPU: the sample that a tile's halo reads (gjxl_amd/csrc/tile_mirror.h) lies
in the line for every extent, and is the mirrored one wherever an output can
need it.

Compiles the product header for the host with g++ and walks over every tile
and tile position of the kernels that use it: the opsin dynamics (64x16 tiles,
halo 2, planes of 8 pixels and more a side, at the full scale and at the half
scale, which is read from the full one at twice the coordinate) and the loop
filters (64x16 tiles, halo 4, planes of 4 pixels and more).
"""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "tile_mirror.h"

// the reflections one after another, for any coordinate
static int Mirror(int c, int size) {
  while (c < 0 || c >= size) c = c < 0 ? -c - 1 : 2 * size - 1 - c;
  return c;
}

static long long n = 0, outside = 0, wrong = 0;

// every position of every tile of a line of `size` samples; with `full` the
// line is formed from one of that many samples, at 2c and 2c + 1
static void Line(int size, int tile, int halo, int full) {
  for (int begin = 0; begin < size; begin += tile) {
    for (int k = 0; k < tile + 2 * halo; ++k) {
      const int c = begin - halo + k, m = gjxl_amd::TileMirror(c, size);
      ++n;
      if (m < 0 || m >= size) ++outside;
      if (full > 0) {
        const int second = 2 * m + 1 < full ? 2 * m + 1 : 2 * m;
        if (2 * m < 0 || 2 * m >= full || second >= full) ++outside;
      }
      // an output lies in the line: it reads no further than the halo
      if (c < size + halo && m != Mirror(c, size)) ++wrong;
    }
  }
}

int main() {
  for (int size = 4; size <= 1100; ++size) {
    for (int tile : {64, 16}) {
      Line(size, tile, 4, 0);
      if (size < 8) continue;
      Line(size, tile, 2, 0);
      Line(size, tile, 2, 2 * size);
      Line(size, tile, 2, 2 * size - 1);
    }
  }
  std::printf("%lld %lld %lld\n", n, outside, wrong);
  return 0;
}
"""


def test_tile_positions_read_samples_of_the_line(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++20", "-I", str(ROOT / "gjxl_amd" / "csrc"), str(src),
                    "-o", str(exe)], check=True)
    n, outside, wrong = map(int, subprocess.run([str(exe)], check=True, capture_output=True,
                                                text=True).stdout.split())
    assert n > 1_000_000
    assert outside == 0
    assert wrong == 0
