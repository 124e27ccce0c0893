// What the FP8 GEMM decides by plain arithmetic: where its large-tile kernel reads. No HIP
// header is needed, so that a host program can check it.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define MIQ_PLAN_FN __host__ __device__ inline
#else
#define MIQ_PLAN_FN inline
#endif

namespace miq {

// Operands read through buffer descriptors end below this many bytes; kFp8Outside lies past every
// such buffer by itself, whatever else is added to it (below 2 GiB).
constexpr int64_t kFp8BufferLimit = 0x7fffff00LL;
constexpr int kFp8Outside = 0x7ffffff0;

// The large-tile kernel's loads: a stage of 64 k is 16-row loads of 64 lanes x 16 bytes, lane l
// taking row l / 4 and 16-byte chunk (l & 3) ^ ((l >> 4) & 3) of its load.
constexpr int kFp8LoadRows = 16;

// Vector offset of one lane's part of load `q` of a tile that begins at row `row0`, in an operand of
// `rows` rows of K bytes; the stage's k (a multiple of 64 below K) is the scalar offset. The row is
// in the vector offset so that the rows past the end, which a tile has whenever its height does
// not divide `rows`, are outside the buffer on their own: with the row in the scalar offset the
// hardware compares the vector offset with (size - scalar offset), which is negative, and as an
// unsigned number huge, once the tile's last rows lie more than `rows` rows into it.
MIQ_PLAN_FN int fp8_large_offset(int row0, int q, int lane, int rows, int K) {
  const int row = row0 + q * kFp8LoadRows + (lane >> 2);
  return row < rows ? row * K + (((lane & 3) ^ ((lane >> 4) & 3)) << 4) : kFp8Outside;
}

}  // namespace miq
