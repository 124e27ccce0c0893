// INT8 weight x bf16 activation GEMM in large blocks, gfx950: long prefill linears and the
// expert GEMMs of a MoE layer over many tokens.
//
//   acc[m, n] = sum_k x[m, k] * q[n, k],  x bf16, q int8 (exact in bf16)
//
// A workgroup of eight wavefronts (two per SIMD) owns a block of 32 MT WM activation rows x
// 64 (8 / WM) weight rows, WM x 8 / WM wavefronts of 32 MT x 64 each on
// v_mfma_f32_32x32x16_bf16. Both operands go from memory straight to LDS (buffer_load ... lds)
// through a ring of three stages of 64 k: the activations as bf16 rows of 128 bytes, the
// weights as raw int8 rows of 64 bytes, 48 KiB a stage. Each wavefront converts its own weight
// fragments to bf16 in registers when it multiplies them (12 VALU instructions per 8 codes,
// every code converted WM times per workgroup, behind the other wavefront's MFMAs), so LDS
// holds one byte per weight and nothing is written to it by the wavefronts.
//
// What bounds it: per 64-k stage a 256 x 256 block takes 2048 clocks of MFMA per SIMD, 208 KiB
// of LDS traffic and 48 KiB from L2 (the 128-row blocks of the wide kernel pull 80 KiB per
// 128 k for half the products, at which L2 and the texture units set its pace). At 12288 x 4096,
// M = 4096 it runs at 1230 TFLOP/s, where this card's library GEMM at its best size reaches
// 1400 (power); a single round of blocks is bound by the ring's latency, about 0.85 us a stage.
//
// LDS: activation row R holds its 16-byte chunk c at position c ^ ((R >> 1) & 7), weight row R
// chunk c at c ^ ((R >> 2) & 3), so that 16 lanes reading one chunk of 16 rows hit the 16
// different 16-byte columns of the 64 banks (swizzled for 32 banks, half of the LDS cycles were
// conflicts); a load writes 64 lanes x 16 bytes contiguously, so each lane fetches the global chunk
// that belongs at its position. k order: sub-step 2 j + e takes k = 32 j + 16 h + 8 e + 0..7 in
// lane half h from both operands (one 16-byte weight read serves two sub-steps).
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "miq_common.h"
#include "wo_block.h"
#include "wo_core.h"
#include "wo_wide.h"

namespace miq {
namespace {

using namespace wo;

enum { BLK_LINEAR = 0, BLK_GATE_UP = 1, BLK_DOWN = 2 };
constexpr int kBK = 64;                       // k per stage
constexpr int kStages = 3;
constexpr int kMoeMT = kMoeTileRows / 32;     // largest row tile of the expert GEMMs, in 32 rows
// bytes of a stage's activations and of the whole stage (WM = 2: 256 + 256 rows, WM = 1: up to
// 160 + 512)
template <int WM>
constexpr int kXBytes = WM == 2 ? 256 * 128 : 32 * kMoeMT * 128;
template <int WM>
constexpr int kStageBytes = kXBytes<WM> + 64 * (8 / WM) * 64;
constexpr int kOutB = 0x7f000000;             // outside every buffer, also with a k offset added
constexpr int kBlkThreads = 512;


struct BlockParams {
  const uint16_t* x;
  int64_t ldx;
  int xbytes;
  const uint8_t* w;
  int wbytes, K;
  const void* scale;
  int M, N;            // linear: rows and columns; MoE: N = I (gate/up) or H (down)
  uint16_t* y;         // linear: [M, N]; gate/up: hbuf [rows, I]; down: ypair [pairs, H]
  int64_t ldy;
  bool vec_store;      // 16-byte stores to y rows
  // linear: tiles_m x tiles_n blocks, the last `halved` of them as two blocks of half the rows
  int tiles_m, tiles_n, full, halved;
  // MoE
  const MoeTile* tiles;
  const int32_t* num_tiles;
  const int32_t* sorted_ids;
  int topk, num_pairs;
  const void* topk_w;
  int w_dtype;
};

template <int N>
__device__ inline void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ inline float bf16r(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// One block: MT 32-row activation tiles per wavefront, WM wavefronts along the rows.
//   m0: first activation row (linear) or first row of the padded expert layout (MoE)
//   nb: column block
template <int MODE, int SD, int WM, int MT>
__device__ inline void block(const BlockParams& p, uint8_t* smem, int m0, int nb, int expert) {
  constexpr int WN = 8 / WM;
  constexpr int kXBlocks = 4 * MT * WM;            // 1-KiB blocks (8 rows) of activations per stage
  constexpr int kWBlocks = 4 * WN;                 // 1-KiB blocks (16 rows) of weights per stage
  constexpr int nX = (kXBlocks + 7) / 8, nW = kWBlocks / 8;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wv / WN, wn = wv - wm * WN;
  const int l32 = lane & 31, h = lane >> 5;

  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), 0, p.xbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), 0, p.wbytes, 0x00020000);
  // this lane's part of this wavefront's loads (a block count below eight is loaded more than
  // once, the same bytes to the same place, so that every wavefront has the same loads in flight)
  int xoff[nX], xdst[nX], woff[nW], wdst[nW];
#pragma unroll
  for (int u = 0; u < nX; ++u) {
    const int b = (wv * nX + u) % kXBlocks;
    const int row = 8 * b + (lane >> 3);
    int src;  // activation row, < 0: none
    if (MODE == BLK_LINEAR) {
      src = m0 + row < p.M ? m0 + row : -1;
    } else if (MODE == BLK_GATE_UP) {
      const int pair = p.sorted_ids[m0 + row];
      src = pair < p.num_pairs ? pair / p.topk : -1;
    } else {
      src = m0 + row;
    }
    xoff[u] = src >= 0 ? (int)(src * p.ldx * 2) + (((lane & 7) ^ ((row >> 1) & 7)) << 4) : kOutB;
    xdst[u] = b * 1024;
  }
#pragma unroll
  for (int u = 0; u < nW; ++u) {
    const int b = wv * nW + u;
    const int row = 16 * (b & 3) + (lane >> 2);  // of the 64 of wavefront column b / 4
    int n;                                       // weight row, < 0: none
    if (MODE == BLK_GATE_UP) {  // 32 gate rows, then the 32 up rows of the same columns
      const int c = (nb * WN + (b >> 2)) * 32 + (row & 31);
      n = c < p.N ? (expert * 2 + (row >> 5)) * p.N + c : -1;
    } else {
      const int c = (nb * WN + (b >> 2)) * 64 + row;
      n = c < p.N ? (MODE == BLK_DOWN ? expert * p.N + c : c) : -1;
    }
    woff[u] = n >= 0 ? n * p.K + (((lane & 3) ^ ((row >> 2) & 3)) << 4) : kOutB;
    wdst[u] = kXBytes<WM> + b * 1024;
  }
  // this wavefront's loads u = part, part + parts, ... of stage s into ring slot `slot` (zeros, and
  // no memory traffic, past the last stage: every stage has the same loads in flight)
  const int nst = p.K / kBK;
  auto issue = [&](int s, int slot, int part, int parts) {
    uint8_t* base = smem + slot * kStageBytes<WM>;
    const uint32_t kx = s < nst ? (uint32_t)s * (kBK * 2) : (uint32_t)kOutB, kw = s < nst ? (uint32_t)s * kBK : (uint32_t)kOutB;
#pragma unroll
    for (int u = 0; u < nX + nW; ++u) {
      if (u % parts != part) continue;
      if (u < nX)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (lds_ptr)(base + xdst[u]), 16, (int)((uint32_t)xoff[u] + kx), 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, (lds_ptr)(base + wdst[u - nX]), 16,
                                                 (int)((uint32_t)woff[u - nX] + kw), 0, 0, 0);
    }
  };

  f32x16 acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][t][v] = 0.f;

  // this lane's LDS offsets in a stage: weight pieces of half stage j, activation chunks of
  // sub-step c = 2 j + e
  const int xrow = (wm * 32 * MT + l32) * 128, wrow = kXBytes<WM> + (wn * 64 + l32) * 64;
  int wad[2], xad[4];
#pragma unroll
  for (int j = 0; j < 2; ++j) wad[j] = wrow + (((2 * j + h) ^ ((l32 >> 2) & 3)) << 4);
#pragma unroll
  for (int c = 0; c < 4; ++c) xad[c] = xrow + (((4 * (c >> 1) + 2 * h + (c & 1)) ^ ((l32 >> 1) & 7)) << 4);
  // Fragments are read one sub-step ahead of their MFMAs (two register sets), the last
  // sub-step's MFMAs of a stage run after the next stage's barrier and first reads, and the
  // conversion of the next weights is spread between the MFMAs: the two wavefronts of a SIMD
  // leave the barrier together, so neither covers the other's LDS latency or conversions.
  bf16x8 xf[2][MT], wf[2][2];
  i32x4 wraw[2];
#pragma unroll
  for (int i = 0; i < MT; ++i) xf[1][i] = __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));
#pragma unroll
  for (int t = 0; t < 2; ++t) wf[1][t] = __builtin_bit_cast(bf16x8, make_uint4(0u, 0u, 0u, 0u));
  auto read_w = [&](int base, int j) {
#pragma unroll
    for (int t = 0; t < 2; ++t) wraw[t] = *reinterpret_cast<const i32x4*>(smem + base + wad[j] + t * 2048);
  };
  auto read_x = [&](int base, int c) {
#pragma unroll
    for (int i = 0; i < MT; ++i) xf[c & 1][i] = *reinterpret_cast<const bf16x8*>(smem + base + xad[c] + i * 4096);
  };
  auto multiply = [&](int c) {  // sub-step c's products
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[c & 1][t], xf[c & 1][i], acc[i][t], 0, 0, 0);
  };
  auto convert = [&](int c) {  // sub-step c's weights
#pragma unroll
    for (int t = 0; t < 2; ++t) wf[c & 1][t] = bf16_of_i8((uint32_t)wraw[t][2 * (c & 1)], (uint32_t)wraw[t][2 * (c & 1) + 1]);
  };
  auto interleave = [&] {  // MFMAs with the next weights' conversion between them
#pragma unroll
    for (int q = 0; q < 2 * MT; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x2, 24 / (2 * MT), 0);  // VALU
    }
  };
  issue(0, 0, 0, 1);
  issue(1, 1, 0, 1);
  int slot = 0, free_slot = 2;
  for (int s = 0; s < nst; ++s) {
    // this wavefront's loads of stage s have landed (those of stage s + 1 may be in flight);
    // after the barrier everyone's have, and stage s - 1's slot is free. The next loads go out
    // a few at a time between the sub-steps: all at once they filled the address units' queue
    // and the wavefront's MFMAs waited behind them.
    wait_loads<nX + nW>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int base = slot * kStageBytes<WM>, fill = free_slot;
    slot = slot == kStages - 1 ? 0 : slot + 1;
    free_slot = free_slot == kStages - 1 ? 0 : free_slot + 1;
    read_w(base, 0);
    read_x(base, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(3);  // the stage before's (zeros in the first stage)
    convert(0);
    interleave();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      read_x(base, c + 1);
      issue(s + 2, fill, c, 3);
      __builtin_amdgcn_sched_barrier(0);
      multiply(c);
      convert(c + 1);
      interleave();
      if (c == 0) read_w(base, 1);  // after convert(1), the last use of the first half's weights
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  multiply(3);

  // epilogue: acc[i][t][4 g + v] belongs to row 32 i + lane % 32 and column 32 t + 8 g + 4 h + v of
  // the wavefront's tile. The bf16 results go through LDS, 32 rows at a time (the ring is free
  // once every wavefront is past its last stage), and out as 16-byte pieces of rows.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  constexpr int kCols = MODE == BLK_GATE_UP ? 32 : 64;  // output columns of the wavefront
  constexpr int kPitch = kCols + 8;
  constexpr int kTiles = MODE == BLK_GATE_UP ? 1 : 2;
  uint16_t* ct = reinterpret_cast<uint16_t*>(smem) + wv * (32 * kPitch);
  const int c0 = (nb * WN + wn) * kCols;  // first output column of the wavefront
  // int8_wo.linear's result: bf16(bf16(x @ q^T) * bf16(scale)) (int8_wo.py:17-21)
  auto row_scale = [&](int64_t n) -> float { return bf16r(sd_to_f32<SD>(load_sd_raw<SD>(p.scale, n))); };
  float sc[kTiles][16], su[MODE == BLK_GATE_UP ? 16 : 1];
#pragma unroll
  for (int t = 0; t < kTiles; ++t)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int n = min(c0 + 32 * t + 8 * (v >> 2) + 4 * h + (v & 3), p.N - 1);
      const int64_t r0 = MODE == BLK_LINEAR ? n : MODE == BLK_DOWN ? (int64_t)expert * p.N + n : (int64_t)expert * 2 * p.N + n;
      sc[t][v] = row_scale(r0);
      if (MODE == BLK_GATE_UP) su[v] = row_scale(r0 + p.N);
    }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int mi = m0 + 32 * (wm * MT + i);
    float wt = 1.f;
    if (MODE == BLK_DOWN) {
      const int pair = p.sorted_ids[mi + l32];
      wt = pair < p.num_pairs ? load_scalar(p.topk_w, p.w_dtype, pair) : 0.f;
    }
#pragma unroll
    for (int t = 0; t < kTiles; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        uint32_t o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float f = bf16r(acc[i][t][4 * g + v]) * sc[t][4 * g + v];
          if (MODE == BLK_GATE_UP) {
            const float gt = bf16r(f), up = bf16r(bf16r(acc[i][1][4 * g + v]) * su[4 * g + v]);
            f = bf16r(gt / (1.f + __expf(-gt))) * up;
          } else if (MODE == BLK_DOWN) {
            f = bf16r(f) * wt;
          }
          o[v] = f32_to_bf16(f);
        }
        *reinterpret_cast<uint2*>(ct + l32 * kPitch + 32 * t + 8 * g + 4 * h) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (only this wavefront reads its part)
    constexpr int kPieces = kCols / 8;  // 16-byte pieces per row
#pragma unroll
    for (int u = 0; u < 32 * kPieces / 64; ++u) {
      const int e = lane + 64 * u, row = e / kPieces, col = (e - row * kPieces) * 8;
      const uint4 v = *reinterpret_cast<const uint4*>(ct + row * kPitch + col);
      const int mr = mi + row;
      int64_t dst = mr;
      bool ok = c0 + col < p.N;
      if (MODE == BLK_LINEAR) ok = ok && mr < p.M;
      if (MODE == BLK_DOWN) {
        dst = p.sorted_ids[mr];
        ok = ok && dst < p.num_pairs;
      }
      if (!ok) continue;
      uint16_t* yp = p.y + dst * p.ldy + c0 + col;
      if (p.vec_store) {
        *reinterpret_cast<uint4*>(yp) = v;
      } else {
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          yp[2 * q] = (uint16_t)w4[q];
          yp[2 * q + 1] = (uint16_t)(w4[q] >> 16);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next rows overwrite them
  }
}

template <int SD>
__global__ void __launch_bounds__(kBlkThreads, 2) wo_block_linear_kernel(BlockParams p) {
  extern __shared__ __align__(16) uint8_t smem[];
  // workgroup id % 8 is the XCD: each takes a contiguous run of blocks, activation rows
  // fastest, so the workgroups of one XCD share weight panels and activations in its L2
  int bid = blockIdx.x;
  const bool half = p.halved && bid >= p.full;
  const int count = half ? 2 * p.halved : p.full;
  if (half) bid -= p.full;
  const int xcd = bid & 7, local = bid >> 3;
  const int item = (int)((int64_t)count * xcd / 8) + local;
  if (item >= (int)((int64_t)count * (xcd + 1) / 8)) return;
  const int tile = half ? p.full + item / 2 : item;
  const int tn = tile / p.tiles_m, tm = tile - tn * p.tiles_m;
  if (half) block<BLK_LINEAR, SD, 2, 2>(p, smem, tm * 256 + (item & 1) * 128, tn, 0);
  else block<BLK_LINEAR, SD, 2, 4>(p, smem, tm * 256, tn, 0);
}

template <int MODE, int SD>
__global__ void __launch_bounds__(kBlkThreads, 2) moe_block_kernel(BlockParams p) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int nbs = (p.N + (MODE == BLK_GATE_UP ? 255 : 511)) / (MODE == BLK_GATE_UP ? 256 : 512);
  const int count = *p.num_tiles * nbs;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int item = (int)((int64_t)count * xcd / 8) + local;
  if (item >= (int)((int64_t)count * (xcd + 1) / 8)) return;
  const MoeTile t = p.tiles[item / nbs];
  const int nb = item % nbs;
  switch (t.blocks) {
    case 1: block<MODE, SD, 1, 1>(p, smem, t.row0, nb, t.expert); break;
    case 2: block<MODE, SD, 1, 2>(p, smem, t.row0, nb, t.expert); break;
    case 3: block<MODE, SD, 1, 3>(p, smem, t.row0, nb, t.expert); break;
    case 4: block<MODE, SD, 1, 4>(p, smem, t.row0, nb, t.expert); break;
    default: block<MODE, SD, 1, kMoeMT>(p, smem, t.row0, nb, t.expert); break;
  }
}

template <class K>
void allow_lds(K kernel, std::once_flag& once) {
  std::call_once(once, [&] { allow_max_dynamic_lds(reinterpret_cast<const void*>(kernel)); });
}

template <int SD>
void launch_linear(const BlockParams& p, unsigned grid, hipStream_t st) {
  static std::once_flag once;
  allow_lds(&wo_block_linear_kernel<SD>, once);
  hipLaunchKernelGGL(wo_block_linear_kernel<SD>, dim3(grid), dim3(kBlkThreads), kStages * kStageBytes<2>, st, p);
}

template <int MODE, int SD>
void launch_moe(const BlockParams& p, unsigned grid, hipStream_t st) {
  static std::once_flag once;
  allow_lds(&moe_block_kernel<MODE, SD>, once);
  hipLaunchKernelGGL((moe_block_kernel<MODE, SD>), dim3(grid), dim3(kBlkThreads), kStages * kStageBytes<1>, st, p);
}

}  // namespace

namespace {
bool fits(int64_t M, int64_t N, int64_t K, int64_t ldx) {
  return M * ldx * 2 < kOutB && N * K < kOutB && K < (1 << 22) && M >= 1 && N >= 1 && K >= 128 && K % 128 == 0;
}
}  // namespace

// A launch of T 256 x 256 blocks on 256 CUs (one workgroup each) costs two units per full round
// and, for a last round of at most 128 blocks (run as halves), one; a unit takes 0.83 us per
// 64-k stage. It is compared with the wide plan's modelled time plus 4 us + 0.35 us per MB of
// packed activations for its pack and clear launches; below the wide kernel's range (too few
// tiles to fill the GPU) the prefill kernel stays. Where the line lies comes from a sweep of seven
// N x K (2560 x 4096 .. 19456 x 2560 and 4096 x 12288) at M = 256 .. 3000, by the two models' ratio:
//   wide without K splits, two or three row tiles: the block was faster at every ratio seen (0.8
//     .. 1.33), by 8 to 37 % (19456 x 2560 M = 1024 / 2048 109 / 187 against 130 / 249 us, ratio
//     1.02 / 0.90; 6144 x 2560 M = 1536 56 / 68, 1.29; 4096 x 12288 M = 3000 262 / 284, 1.24);
//   one row tile or K splits: faster or even up to 1.13 (6144 x 2560 M = 512 34 / 37, 1.13; 2560 x
//     9728 M = 2048 111 / 135, 0.99; 4096 x 12288 M = 1280 139 / 162, 1.07), slower from 1.15 up
//     (12288 x 4096 M = 256 50 / 47, 1.15; 2560 x 9728 M = 1536 / 1024 106 / 101, 1.32, and 103 / 77,
//     1.77);
//   one row tile at a deep K: even at 1.07, slower from there (a second sweep of nine N, seven K and 22
//     M: at K = 2560 the block took 0.85 to 0.98 of the wide kernel's time up to 1.14, at K = 4096
//     0.85 to 0.94 up to 1.06 and 0.92 to 1.08 past it; 6144 x 4096 M = 450 47.8 / 45.0, 1.14).
bool wo_block_planned(int64_t M, int64_t N, int64_t K, int64_t ldx, const WidePlan& wide) {
  const Tuning& t = tuning();
  if (t.wo_block == 0 || !fits(M, N, K, ldx)) return false;
  if (t.wo_block == 1) return true;
  // switches that force a plan of the other prefill kernels
  if (wide.mt == 0 || t.wo_wide_mt >= 0 || t.wo_wide_s > 0 || t.wo_prefill_s > 0) return false;
  const int64_t T = ((M + 255) / 256) * ((N + 255) / 256), rest = T % 256;
  const int64_t units = 2 * (T / 256) + (rest == 0 ? 0 : rest <= 128 ? 1 : 2);
  const double block_us = 4.0 + 0.83 * (double)(units * (K / kBK));
  const double wide_us = wide.us + 4.0 + 0.35e-6 * (double)wide.pack_bytes;
  const double line = wide.S == 1 && wide.mt >= 2 ? 1.35 : wide.S == 1 && K >= 3584 ? 1.06 : 1.14;
  return block_us < line * wide_us;
}

int wo_block_launch(const uint16_t* x, int64_t ldx, const uint8_t* w, const void* scale, int sd, uint16_t* y, int64_t ldy,
                    int64_t M, int N, int K, hipStream_t st, const char* name) {
  MIQ_REQUIRE(fits(M, N, K, ldx), "%s: operands too large for the block kernel", name);
  BlockParams p{};
  p.x = x;
  p.ldx = ldx;
  p.xbytes = (int)(((M - 1) * ldx + K) * 2);
  p.w = w;
  p.wbytes = (int)((int64_t)N * K);
  p.K = K;
  p.scale = scale;
  p.M = (int)M;
  p.N = N;
  p.y = y;
  p.ldy = ldy;
  p.vec_store = (reinterpret_cast<uintptr_t>(y) & 15) == 0 && ldy % 8 == 0;
  p.tiles_m = (int)((M + 255) / 256);
  p.tiles_n = (N + 255) / 256;
  const int T = p.tiles_m * p.tiles_n, rest = T % 256;
  // a last round of at most 128 blocks leaves half the CUs idle: those blocks run as two halves
  p.halved = rest <= 128 ? rest : 0;
  p.full = T - p.halved;
  // every XCD's share of the full and of the half blocks fits (with halves, full is a multiple
  // of 256)
  const unsigned grid = (unsigned)((p.full + 7) / 8 * 8 + (2 * p.halved + 7) / 8 * 8);
  if (sd == MIQ_BF16) launch_linear<MIQ_BF16>(p, grid, st);
  else if (sd == MIQ_F16) launch_linear<MIQ_F16>(p, grid, st);
  else launch_linear<MIQ_F32>(p, grid, st);
  return check_launch(name);
}

bool moe_block_fits(int64_t T, int64_t topk, int64_t E, int64_t H, int64_t I, int64_t max_rows) {
  return H % 128 == 0 && I % 128 == 0 && T * H * 2 < kOutB && max_rows * I * 2 < kOutB && E * 2 * I * H < kOutB &&
         H < (1 << 22) && I < (1 << 22);
}

int moe_block_launch(const MoeBlockArgs& a, hipStream_t st, const char* name) {
  BlockParams p{};
  p.tiles = a.tiles;
  p.num_tiles = a.num_tiles;
  p.sorted_ids = a.sorted_ids;
  p.topk = a.topk;
  p.num_pairs = a.T * a.topk;
  p.topk_w = a.topk_w;
  p.w_dtype = a.w_dtype;
  p.vec_store = true;
  const int64_t max_tiles = (int64_t)p.num_pairs / kMoeTileRows + std::min(a.E, p.num_pairs);
#define MIQ_MOE_BLOCK(MODE_, BN_)                                                                          \
  do {                                                                                                     \
    const unsigned grid = (unsigned)((max_tiles * ((p.N + BN_ - 1) / BN_) + 7) / 8 * 8 + 8);              \
    if (a.sd == MIQ_BF16) launch_moe<MODE_, MIQ_BF16>(p, grid, st);                                        \
    else if (a.sd == MIQ_F16) launch_moe<MODE_, MIQ_F16>(p, grid, st);                                     \
    else launch_moe<MODE_, MIQ_F32>(p, grid, st);                                                          \
  } while (0)
  p.x = a.hidden;
  p.ldx = a.H;
  p.xbytes = (int)((int64_t)a.T * a.H * 2);
  p.w = a.gu_q;
  p.wbytes = (int)((int64_t)a.E * 2 * a.I * a.H);
  p.K = a.H;
  p.scale = a.gu_s;
  p.N = a.I;
  p.y = a.hbuf;
  p.ldy = a.I;
  MIQ_MOE_BLOCK(BLK_GATE_UP, 256);
  p.x = a.hbuf;
  p.ldx = a.I;
  p.xbytes = (int)(a.max_rows * a.I * 2);
  p.w = a.dn_q;
  p.wbytes = (int)((int64_t)a.E * a.H * a.I);
  p.K = a.I;
  p.scale = a.dn_s;
  p.N = a.H;
  p.y = a.ypair;
  p.ldy = a.H;
  MIQ_MOE_BLOCK(BLK_DOWN, 512);
#undef MIQ_MOE_BLOCK
  return check_launch(name);
}

}  // namespace miq
