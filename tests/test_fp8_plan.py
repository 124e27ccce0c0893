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
// their row and chunk. `split`: the load's row in the scalar offset, the k in the vector offset.
extern "C" long faults(int rows, int K, int tile, int loads, int split) {
  const uint32_t size = (uint32_t)rows * (uint32_t)K;
  const int row0 = (rows - 1) / tile * tile;
  long bad = 0;
  for (int k0 : {0, 64, K - 64})
    for (int q = 0; q < loads; ++q)
      for (int lane = 0; lane < 64; ++lane) {
        const int row = row0 + 16 * q + lane / 4, chunk = (lane & 3) ^ ((lane >> 4) & 3);
        Load l{(uint32_t)fp8_large_offset(row0, q, lane, rows, K), (uint32_t)k0};
        if (split) l = Load{(uint32_t)(fp8_large_offset(row0, 0, lane, rows, K) + k0), (uint32_t)(16 * q * K)};
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

extern "C" int whole(int rows, int tile) { return fp8_whole_tiles(rows, tile); }

extern "C" int kernel(long M, long N, long K, int buffers, int rows16) {
  return (int)fp8_plan(M, N, K, buffers, rows16).kernel;
}
"""
SPLIT, LARGE, SMALL, PREVIOUS = range(4)


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("fp8_plan")
    src, so = str(d / "harness.cpp"), str(d / "harness.so")
    with open(src, "w") as f:
        f.write(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, src, "-o", so], check=True)
    out = ctypes.CDLL(so)
    out.faults.restype = ctypes.c_long
    out.kernel.argtypes = [ctypes.c_long] * 3 + [ctypes.c_int] * 2
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
def test_rows_go_into_the_scalar_offset_only_with_whole_tiles(lib, tile, loads):
    """Operands of whole tiles may have the row in the scalar part, up to the largest one; the
    check refuses that for every other number of rows, which the rule keeps from it."""
    for tiles in (1, 2, 11):
        assert lib.whole(tiles * tile, tile) and lib.faults(tiles * tile, 2560, tile, loads, 1) == 0
    last = 0x7fffff00 // 128 // tile * tile
    assert lib.whole(last, tile) and lib.faults(last, 128, tile, loads, 1) == 0
    for rows in (1, 65, 129, 175, tile - 1, tile + 1, 5 * tile + 64):
        assert not lib.whole(rows, tile) and lib.faults(rows, 2560, tile, loads, 1) > 0, rows


# (M, N, K) -> the kernel that measures fastest there, of every size by more than 5 %
FASTEST = {(1, 6144, 2560): SPLIT, (64, 2560, 9728): SPLIT, (512, 2560, 4096): SPLIT, (100, 2560, 4096): SPLIT,
           (200, 19456, 2560): LARGE, (300, 19456, 2560): LARGE, (1000, 19456, 2560): LARGE,
           (2048, 6144, 2560): LARGE, (1280, 6144, 4096): LARGE, (2560, 6144, 4096): LARGE, (1280, 12288, 4096): LARGE,
           (1536, 4608, 9728): LARGE, (2048, 3264, 3200): LARGE, (2560, 2560, 4096): LARGE, (1024, 8192, 8192): LARGE}


def test_the_fastest_kernel_is_chosen(lib):
    for size, kernel in FASTEST.items():
        assert lib.kernel(*size, 1, 1) == kernel, size


def test_the_large_tiles_replacements_stay_with_calls_they_cannot_take(lib):
    """Over a grid of sizes: a call with 16-byte output rows and operands in reach of buffer
    descriptors runs on split or large tiles, whatever divides N; one without runs on split or
    on register-staged tiles, of 256 x 192 only where it always did."""
    seen = set()
    for M in list(range(1, 66, 8)) + list(range(65, 4200, 61)):
        for N in (16, 192, 200, 1008, 1920, 2560, 3264, 4608, 6144, 12288, 19456, 20736):
            for K in (128, 256, 2560, 4096, 9728):
                assert lib.kernel(M, N, K, 1, 1) in (SPLIT, LARGE), (M, N, K)
                others = PREVIOUS if M >= 1024 and N % 192 == 0 else SMALL
                assert lib.kernel(M, N, K, 1, 0) in (SPLIT, others), (M, N, K)
                assert lib.kernel(M, N, K, 0, 1) == others, (M, N, K)
                seen |= {lib.kernel(M, N, K, 1, 1), lib.kernel(M, N, K, 1, 0)}
            assert lib.kernel(M, N + 4, 2560, 1, 1) in (SPLIT, SMALL), (M, N + 4)  # (rows of 8 outputs)
    assert seen == {SPLIT, LARGE, SMALL, PREVIOUS}


def test_the_gpu_tests_reach_every_kernel(lib):
    """The sizes of the GPU tests, by the kernel that serves them."""
    import test_gpu_fp8_split as split
    import test_gpu_gemm as gemm
    by = {}
    for size in split.SIZES:
        for rows16 in (1, 0):  # (the padded outputs rule out 16-byte rows)
            by.setdefault(lib.kernel(*size, 1, rows16), []).append(size)
    assert len(by[SPLIT]) > 10
    assert {M for M, _, _ in by[LARGE]} >= {129, 200, 239, 255, 257, 20000}
    assert len(by[SMALL]) >= 3 and len(by[PREVIOUS]) >= 1
    assert lib.kernel(*gemm.FP8_VARIANT_SIZE, 1, 1) == LARGE and lib.kernel(*gemm.FP8_VARIANT_SIZE, 1, 0) == PREVIOUS
    assert lib.kernel(*gemm.FP8_SMALL_SIZE, 0, 1) == SMALL
