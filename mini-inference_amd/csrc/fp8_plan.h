// What the FP8 GEMM decides by plain arithmetic: the kernel of a call, and where the large-tile
// kernel reads. No HIP header is needed, so that a host program can check it.
#pragma once
#include <algorithm>
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

// Whether tiles of `tile` rows cover an operand of `rows` rows without rows past its end. The scalar
// offset of such an operand's loads may hold the load's row (q * kFp8LoadRows * K): it stays inside
// the buffer, and so does its sum with the vector offset of load 0.
MIQ_PLAN_FN bool fp8_whole_tiles(int rows, int tile) { return rows % tile == 0; }

// Vector offset of one lane's part of load `q` of a tile that begins at row `row0`, in an operand of
// `rows` rows of K bytes; the stage's k (a multiple of 64 below K) is the scalar offset. The row is
// in the vector offset so that the rows past the end of an operand that its tiles do not cover
// evenly are outside the buffer on their own: with the row in the scalar offset the hardware
// compares the vector offset with (size - scalar offset), which is negative, and as an unsigned
// number huge, once the tile's last rows lie more than `rows` rows into it.
MIQ_PLAN_FN int fp8_large_offset(int row0, int q, int lane, int rows, int K) {
  const int row = row0 + q * kFp8LoadRows + (lane >> 2);
  return row < rows ? row * K + (((lane & 3) ^ ((lane >> 4) & 3)) << 4) : kFp8Outside;
}

constexpr int kFp8Step = 128;  // K is a multiple of it

// The split kernel: 16 mt x 16 nt tiles, nw wavefronts per workgroup that split K, and the modelled
// time.
struct Fp8SplitPlan {
  int mt = 0, nt = 0, nw = 0;
  double us = 0.0;
};

// Tile sizes, wavefronts and modelled time of a call. The kernel runs at the rate at which a CU pulls
// operands from L2, so the plan takes the tile that needs the fewest bytes on the busiest CU
// (tiles per CU, rounded up, times the tile's rows; activation rows, read 64 bytes at a time,
// weigh 1.3 times the weights' whole lines), and fewer wavefronts per workgroup where a CU
// holds several workgroups. Chosen from a sweep on MI355X of every (MT, NT, NW) below over N x
// K = 6144 x 2560, 2560 x 9728, 19456 x 2560, 2560 x 4096 and 1024 x 1024 at M = 1 .. 1000: the
// plan is within 10 % of the fastest tile. Split against 128 x 128 tiles, us (rotating weight
// copies): 6144 x 2560 M = 1 / 16 / 64 / 256 / 512: 6 / 7 / 11 / 21 / 31 against 31 / 33 / 40 /
// 42 / 41; 2560 x 9728: 8 / 11 / 17 / 31 / 54 against 101 / 102 / 110 / 113 / 110. Modelled
// time (fp8_plan compares it with the other kernels'): 4 us, those bytes at 41 (K = 2560) to
// 59 KB (K = 9728) per us, and 0.1 us per MB of weights.
inline Fp8SplitPlan fp8_split_plan(int64_t M, int64_t N, int64_t K) {
  static const int kTiles[][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}, {2, 4}, {4, 2}, {4, 4}};
  Fp8SplitPlan best;
  double best_bytes = 0.0;
  for (const auto& t : kTiles) {
    const int64_t items = ((M + 16 * t[0] - 1) / (16 * t[0])) * ((N + 16 * t[1] - 1) / (16 * t[1]));
    const int64_t per_cu = (items + 255) / 256;
    const double bytes = (double)per_cu * (double)K * 16.0 * (1.3 * t[0] + t[1]);
    if (best.mt != 0 && bytes >= best_bytes) continue;
    best_bytes = bytes;
    best.mt = t[0];
    best.nt = t[1];
    best.nw = per_cu == 1 ? 8 : per_cu <= 3 ? 4 : 2;
  }
  const int64_t steps = K / kFp8Step;
  while (best.nw > 2 && steps < 2 * best.nw) best.nw /= 2;
  best.us = 4.0 + best_bytes / (34e3 + 330.0 * (double)std::min<int64_t>(steps, 76)) + 1e-7 * (double)N * (double)K;
  return best;
}

// Large: 256 x 192 tiles on 32x32x64 MFMAs. For calls that it does not take, small: 128 x 128 tiles,
// and previous: 256 x 192 tiles staged through registers.
enum class Fp8Kernel { kSplit, kLarge, kSmall, kPrevious };
struct Fp8Plan {
  Fp8Kernel kernel;
  Fp8SplitPlan split;  // of kSplit
};

// Time of `tiles` tiles that run `per_round` at a time: a fixed part per round, and per k-step
// one that grows with the tiles of the round (they share L2 and memory).
inline double fp8_rounds_us(int64_t tiles, int64_t per_round, double fixed, double steps, double base, double share) {
  const int64_t full = tiles / per_round, rest = tiles % per_round;
  double us = (double)full * (fixed + steps * (base + share));
  if (rest) us += fixed + steps * (base + share * (double)rest / (double)per_round);
  return us;
}

// The kernel of least modelled time. `buffers`: both operands below kFp8BufferLimit; `rows16`:
// y takes 16-byte stores (the large-tile kernel's). Fitted on MI355X over N = 256 .. 28672, K = 512
// .. 9728 and M = 1 .. 4096 (1320 calls, every kernel forced): the choice is the fastest kernel or
// within 5 % of it in all but 28 calls, and none is slower than with large tiles from M = 1024 on
// where 192 divides N and small ones otherwise (the rule before the split kernel). A call that
// takes the large tiles is never faster on the small ones. Split / large / small, us:
//   19456 x 2560  M = 65 25/30/42, 128 34/33/46, 200 47/37/47, 300 61/34/47, 1000 149/76/126
//   6144 x 4096   M = 1280 88/42/55, 2560 172/85/106;   2560 x 4096  M = 512 26/38/48, 2560 86/42/56
//   8192 x 8192   M = 512 88/86/96, 1024 174/89/103;    2560 x 9728  M = 1024 75/82/95
//   12288 x 4096  M = 129 32/41/55, 1280 175/97/119
// (the previous kernel: 71 us at 6144 x 4096, M = 1280, and 140 at 2560). The split model errs high
// for 65 .. 256 rows of a deep K and a wide N (the first of the last row), which run on large
// tiles all the same.
inline Fp8Plan fp8_plan(int64_t M, int64_t N, int64_t K, bool buffers, bool rows16) {
  const bool large = buffers && rows16 && N % 8 == 0;
  const double us =
      large ? fp8_rounds_us(((M + 255) / 256) * ((N + 191) / 192), 256, 7.6, (double)(K / 64), 0.45, 0.25)
            : fp8_rounds_us(((M + 127) / 128) * ((N + 127) / 128), 512, 13.4, (double)(K / kFp8Step), 0.98, 0.48);
  if (buffers) {
    const Fp8SplitPlan split = fp8_split_plan(M, N, K);
    if (split.us < us) return {Fp8Kernel::kSplit, split};
  }
  if (large) return {Fp8Kernel::kLarge, {}};
  return {M >= 1024 && N % 192 == 0 ? Fp8Kernel::kPrevious : Fp8Kernel::kSmall, {}};
}

}  // namespace miq
