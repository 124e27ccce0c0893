"""The FP8 GEMM's host arithmetic (csrc/fp8_plan.h), compiled for the CPU."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "mini-inference_amd", "csrc")

HARNESS = r"""
#include <initializer_list>
#include <cstdint>
#include "fp8_plan.h"
using namespace miq;

// A 16-byte buffer load as the hardware may check it: the vector offset against (size - scalar
// offset), unsigned; against the size alone; or the sum of both against the size.
struct Load { uint32_t voff, soff; };
static bool through(Load l, uint32_t size, int rule) {
  if (rule == 0) return l.voff < size - l.soff;
  if (rule == 1) return l.voff < size;
  return l.voff + l.soff < size;
}

// Lanes of the last tile's loads (`loads` loads of 16 rows) that any rule lets read past the
// operand, that any rule rejects though their row exists, or that read another address than
// their row and chunk. `split`: the row in the scalar offset, the k in the vector offset.
extern "C" long faults(int rows, int K, int tile, int loads, int split) {
  const uint32_t size = (uint32_t)rows * (uint32_t)K;
  const int row0 = (rows - 1) / tile * tile;
  long bad = 0;
  for (int k0 : {0, 64, K - 64})
    for (int q = 0; q < loads; ++q)
      for (int lane = 0; lane < 64; ++lane) {
        const int row = row0 + 16 * q + lane / 4, chunk = (lane & 3) ^ ((lane >> 4) & 3);
        Load l{(uint32_t)fp8_large_offset(row0, q, lane, rows, K), (uint32_t)k0};
        if (split) l = Load{(uint32_t)((row0 + lane / 4) * K + chunk * 16 + k0), (uint32_t)(16 * q * K)};
        for (int rule = 0; rule < 3; ++rule) {
          const bool reads = through(l, size, rule);
          const uint64_t at = (uint64_t)l.voff + l.soff;
          if (reads && at + 16 > size) ++bad;
          else if (row < rows && (!reads || at != (uint64_t)row * K + chunk * 16 + k0)) ++bad;
          else if (row >= rows && reads) ++bad;
        }
      }
  return bad;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("fp8_plan")
    src, so = str(d / "harness.cpp"), str(d / "harness.so")
    with open(src, "w") as f:
        f.write(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, src, "-o", so], check=True)
    out = ctypes.CDLL(so)
    out.faults.restype = ctypes.c_long
    return out


# rows of one part tile and of several; the largest operands that take buffer descriptors
ROWS = [1, 15, 16, 17, 65, 129, 200, 239, 240, 241, 255, 256, 257, 300, 1000, 2048]
TILES = [(256, 16), (192, 12)]


@pytest.mark.parametrize("tile,loads", TILES)
def test_large_tiles_read_inside_their_operands(lib, tile, loads):
    """Activation (256 rows) and weight (192 rows) tiles: rows that exist are read at their
    address and rows past the end not at all, however the range check treats the scalar
    offset."""
    for K in (128, 256, 2560, 9728):
        for rows in ROWS:
            assert lib.faults(rows, K, tile, loads, 0) == 0, (rows, K)
    for K in (128, 1 << 20, 1 << 24):
        rows = 0x7fffff00 // K - 1
        assert lib.faults(rows, K, tile, loads, 0) == 0, (rows, K)


@pytest.mark.parametrize("tile,loads", TILES)
def test_the_check_finds_rows_in_the_scalar_offset(lib, tile, loads):
    """The same check refuses offsets with the row in the scalar part, for operands lower than a
    tile (a planted mistake)."""
    for rows in (1, 65, 129, 175):
        assert lib.faults(rows, 2560, tile, loads, 1) > 0, rows
