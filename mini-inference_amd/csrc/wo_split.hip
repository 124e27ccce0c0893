// INT8 weight x bf16 activation GEMM for decode batches, gfx950:
//
//   y[m, n] = bf16( bf16(sum_k x[m, k] * q[n, k]) * bf16(scale[n]) )
//
// A workgroup owns a tile of 16 MT activation rows x 16 NT weight rows over the whole of K; its
// wavefronts split K and multiply the whole tile over their own k-steps of 128; their fp32 tiles
// are added in LDS in wavefront order. Nothing is shared between the wavefronts before that, so
// the K loop has no barrier: weights go straight to registers four steps ahead (the memory's
// latency under load is several steps long: with one step ahead 2560 x 4096, M = 64 took 14.2 us
// instead of 11.4), activations by loads to LDS into the wavefront's own two step buffers, in whole
// 256-byte row pieces. The codes are converted to bf16 in registers (exact), so there are no
// activation sums. What bounds it: the operand bytes a CU pulls, at about 46 KB per us, and the
// weights' first arrival.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "miq_common.h"
#include "wo_core.h"
#include "wo_split.h"

namespace miq {
namespace {

using namespace wo;

constexpr int kOutS = 0x7ffffff0;  // outside every buffer: the load returns zeros
constexpr int kAhead = 4;  // k-steps of weights in flight

struct WoSplitParams {
  const uint16_t* x;
  int64_t ldx;
  int xbytes;
  const uint8_t* w;
  const void* scale;
  uint16_t* y;
  int64_t ldy;
  int M, N, K;
  int tiles_m, items;
  bool vec_store;  // y rows 8-byte aligned (4 outputs per store)
};


// f(integral_constant 0) .. f(integral_constant kAhead - 1)
template <int I = 0, class F>
__device__ inline void unroll_steps(F&& f) {
  if constexpr (I < kAhead) {
    f(std::integral_constant<int, I>{});
    unroll_steps<I + 1>(f);
  }
}

template <int MT, int NT, int kWaves, int SD>
__global__ void __launch_bounds__(kWaves * 64)
wo_split_kernel(WoSplitParams p) {
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // XCD x (= workgroup id % 8) takes a contiguous eighth of the items, activation tiles
  // fastest, so the workgroups that read one weight tile share an L2
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int item = (int)((int64_t)p.items * xcd / 8) + local;
  if (item >= (int)((int64_t)p.items * (xcd + 1) / 8)) return;
  const int tn = item / p.tiles_m, tm = item - tn * p.tiles_m;
  const int n0 = tn * 16 * NT, m0 = tm * 16 * MT;
  const int steps = p.K / kStepK;
  const int s0 = steps * wv / kWaves, s1 = steps * (wv + 1) / kWaves;  // this wavefront's k-steps

  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), 0, p.N * p.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.x), 0, p.xbytes, 0x00020000);
  // weights: load h covers rows 8 h .. 8 h + 7 of a tile as whole 128-byte lines, in address
  // order within each 64-byte half; lanes_to_mfma turns two loads into the MFMA layout: lane
  // (g, r) then holds codes 16 g .. + 15 of both halves of row r, and of the activations the same k
  const int lrr = (lane >> 2) & 7, lcl = lane & 3, lc2 = lane >> 5;
  const int bp_addr = (32 * (r >> 3) + 4 * (r & 7) + g) * 4;
  int woff[NT][2], xoff[4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int n = n0 + 16 * t + 8 * h + lrr;
      woff[t][h] = n < p.N ? n * p.K + lc2 * 64 + lcl * 16 : kOutS;
    }
  // activations: a load to LDS covers 4 rows x 256 bytes; row R's 16-byte chunk c sits at position
  // c ^ (R & 15), so the 16 rows of a fragment read hit 16 different columns. Rows past M lie
  // past the buffer (zeros).
  const int ldx2 = (int)p.ldx * 2;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    const int row = 4 * b + (lane >> 4);
    xoff[b] = (m0 + row) * ldx2 + (((lane & 15) ^ row) << 4);
  }
  uint8_t* const xbuf = smem + wv * (2 * MT * 4096);  // this wavefront's two step buffers
  uint4 wq[kAhead][NT][2];
  auto request_w = [&](auto set_c, int s) {
    constexpr int d = decltype(set_c)::value;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int off = s < s1 && woff[t][h] != kOutS ? woff[t][h] + s * kStepK : kOutS;
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(wrs, off, 0, 0);
        wq[d][t][h] = *reinterpret_cast<const uint4*>(&v);
      }
  };
  auto request_x = [&](int d, int s) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int off = s < s1 ? xoff[b] + i * 16 * ldx2 + s * (2 * kStepK) : kOutS;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xrs, (lds_ptr)(xbuf + (d * MT + i) * 4096 + b * 1024), 16, off, 0, 0, 0);
      }
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xad[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) xad[j] = r * 256 + (((8 * (j >> 1) + 2 * g + (j & 1)) ^ r) << 4);
  auto multiply = [&](auto set_c) {
    constexpr int d = decltype(set_c)::value;
    // this step's activations have landed (issued after them: one step of weights and one of
    // activations), and with them its weights; the buffers are the wavefront's own, so no barrier
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NT + 4 * MT) : "memory");
    bf16x8 wf[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      uint4 wl[2];
      lanes_to_mfma(bp_addr, wq[d][t][0], wq[d][t][1], wl[0], wl[1]);
      wf[t][0] = bf16_of_i8(wl[0].x, wl[0].y);
      wf[t][1] = bf16_of_i8(wl[0].z, wl[0].w);
      wf[t][2] = bf16_of_i8(wl[1].x, wl[1].y);
      wf[t][3] = bf16_of_i8(wl[1].z, wl[1].w);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x8 xf = *reinterpret_cast<const bf16x8*>(xbuf + ((d & 1) * MT + i) * 4096 + xad[j]);
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][j], xf, acc[t][i], 0, 0, 0);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next loads overwrite them
  };
  unroll_steps([&](auto d_c) { request_w(d_c, s0 + decltype(d_c)::value); });
  request_x(0, s0);
  request_x(1, s0 + 1);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * MT) : "memory");  // the first step's (and the weights before them)
  for (int sb = s0; sb < s1; sb += kAhead) {
    unroll_steps([&](auto d_c) {
      const int s = sb + decltype(d_c)::value;
      if (s >= s1) return;  // uniform
      multiply(d_c);
      request_w(d_c, s + kAhead);
      request_x(decltype(d_c)::value & 1, s + 2);
    });
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // every wavefront is done with its buffers
  f32x4* red = reinterpret_cast<f32x4*>(smem);  // [wavefront][tile][lane]
  // the sum over the wavefronts, in wavefront order
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < MT; ++i) red[(wv * (MT * NT) + t * MT + i) * 64 + lane] = acc[t][i];
  __syncthreads();
  for (int e = tid; e < MT * NT * 64; e += kWaves * 64) {
    const int ti = e >> 6, l = e & 63;
    f32x4 s = red[e];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) s += red[w * (MT * NT) * 64 + e];
    const int t = ti / MT, i = ti - t * MT;
    const int m = m0 + 16 * i + (l & 15), n = n0 + 16 * t + 4 * (l >> 4);
    if (m >= p.M || n >= p.N) continue;  // (N is a multiple of 16)
    uint32_t o[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float sc = bf16_to_f32(f32_to_bf16(sd_to_f32<SD>(load_sd_raw<SD>(p.scale, n + v))));
      o[v] = f32_to_bf16(bf16_to_f32(f32_to_bf16(s[v])) * sc);
    }
    uint16_t* dst = p.y + (int64_t)m * p.ldy + n;
    if (p.vec_store) {
      *reinterpret_cast<uint2*>(dst) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v) dst[v] = (uint16_t)o[v];
    }
  }
}

template <int MT, int NT, int kWaves>
void go(const WoSplitParams& p, int sd, hipStream_t st) {
  const unsigned grid = (unsigned)((p.items + 7) / 8 * 8 + 8);  // every XCD's share fits
  const size_t lds = std::max((size_t)kWaves * 2 * MT * 4096, (size_t)kWaves * MT * NT * 1024);
#define MIQ_WS_GO(SD_)                                                                                          \
  do {                                                                                                          \
    static std::once_flag once;                                                                                 \
    std::call_once(once, [] { allow_max_dynamic_lds(reinterpret_cast<const void*>(&wo_split_kernel<MT, NT, kWaves, SD_>)); }); \
    hipLaunchKernelGGL((wo_split_kernel<MT, NT, kWaves, SD_>), dim3(grid), dim3(kWaves * 64), lds, st, p);              \
  } while (0)
  if (sd == MIQ_BF16) MIQ_WS_GO(MIQ_BF16);
  else if (sd == MIQ_F16) MIQ_WS_GO(MIQ_F16);
  else MIQ_WS_GO(MIQ_F32);
#undef MIQ_WS_GO
}

}  // namespace

// Tile and wavefronts of a call (mt = 0: another kernel). The tile that needs the fewest
// operand bytes on the busiest CU (tiles per CU, rounded up, times 2 bytes per activation and 1
// per weight); eight wavefronts where a CU has one small tile and K is long. From a sweep of
// every tile over N x K = 19456 x 2560, 6144 x 2560, 2560 x 9728, 2560 x 4096, 12288 x 4096 and
// 1024 x 1024 at M = 8 .. 256 (MI355X, rotating weight copies), split / streamed kernel, us:
//   M              8          16         32         48         64
//   6144 x 2560    9.0/11.3   9.3/12.9   10.3/15.7  11.1/23.1  11.3/29.9
//   2560 x 9728    12.2/13.3  13.4/15.3  17.0/23.3  16.9/30.0  19.6/37.1
//   2560 x 4096    7.8/10.3   8.1/11.5   10.1/19.9  10.2/24.6  11.4/30.2
//   12288 x 4096   14.9/16.2  15.2/17.4  16.9/23.5  19.5/29.0  23.0/33.0
//   19456 x 2560   18.0/16.7  18.1/18.2  20.1/22.2  22.6/27.6  26.2/33.0
// The rule's lines come from two more sweeps, of this kernel against the others over N = 512 ..
// 151936, K = 512 .. 19456 and M = 5 .. 256 (5200 calls): inside the lines it was nowhere slower by
// more than 3 %. Each gives the deepest K that a tile shape pays for: a workgroup walks all of K,
// where the streamed kernel gives a deep K to several workgroups, so narrow tiles (few weights
// per activation) lose first. Split / other kernel, us:
//   M = 5 .. 16:  5120 x 12288 M = 8 20.7/17.6, 512 x 16384 13.9/11.1; 12288 x 4096 M = 8 16.2/15.2;
//     M = 5 (a plan of one weight tile is the only one that pays) 6144 x 2560 8.4/7.4;
//   16-row tiles by 64 or 80 weights:  8192 x 4096 M = 17 14.9/19.0, x 8192 25.4/23.6; 6144 x 6144 M
//     = 36 23/24, x 14336 M = 40 47.3/39.9;
//   32-row tiles by 64 or 80:  20480 x 3072 M = 18 22.7/21.2; 9728 x 9728 M = 36 41.9/38.2, M = 60
//     faster.
// Tiles of 32 rows or more fill a CU's LDS, so a second tile waits for the first, whereas the
// other kernels' time grows with the weights alone:
//   two tiles per CU:  by 48 weights 24576 x 2560 M = 32 20.9/26.8; by 64 28672 x 1024 13.7/17.4,
//     32768 x 2048 M = 17 22.6/20.5, 28672 x 8192 M = 48 72/80; by 80 40960 x 2560 M = 17
//     37.4/31.2, x 8192 M = 48 91/130;
//   three:  49152 x 1024 M = 64 33.5/25.6, x 4096 M = 40 73/71, x 8192 106/126;
//   more (a vocabulary's projection):  151936 x 2560 M = 17 137/83, 50304 x 2048 M = 64 58/45.
// Past 64 rows it takes the calls whose modelled time (4 us + the bytes at 46 KB per us + 0.1 us
// per MB of weights) is below what the prefill kernels were never seen under at that depth of K: 26
// us, or 17 us below 20 k-steps (M = 128: 6144 x 2560 15.4 against 33.7 us, 2560 x 4096 13.1
// against 28.6, 1024 x 1024 5.2 against 19.3; 19456 x 2560 44.1 against 37.9, not taken), and with
// a second tile per CU only from 16 k-steps up (M = 96, 12288 x 512 13.8 against 11.3, x 1024 17.7
// against 16.1, x 2560 27.9 against 35.8).
static bool split_is_faster(const WoSplitPlan& pl, int64_t per_cu, double bytes, int64_t M, int64_t N, int64_t K) {
  const int64_t steps = K / kStepK;
  if (M <= 4 || steps > 128) return false;
  if (M > 64) {
    const double us = 4.0 + bytes / 46e3 + 1e-7 * (double)N * (double)K;
    return us < (steps >= 20 ? 26.0 : 17.0) && (per_cu == 1 || steps >= 16);
  }
  if (M < 8) return (pl.nt == 1 && steps <= 64) || (M >= 6 && pl.nt <= 3 && steps <= (pl.nt == 2 ? 32 : 24));
  if (M <= 16) {
    if (pl.nt <= 2) return steps <= (pl.nt == 1 ? 80 : 64);
    return pl.nt == 3 && (per_cu > 1 || M >= 12 || steps <= 24 || steps >= 48);
  }
  if (per_cu == 1) {
    if (pl.nt <= 3 || pl.mt >= 3) return true;
    if (pl.mt == 1) return steps <= (M <= 24 ? 32 : 64);
    return M > 48 || steps <= (pl.nt == 4 ? 80 : M <= 24 ? 20 : 32);
  }
  if (per_cu == 2 && (pl.nt <= 3 || (pl.nt == 4 && steps <= 12) || (pl.nt == 5 && steps >= 32))) return true;
  return M > 24 && steps >= 64 && (per_cu == 2 || (per_cu == 3 && pl.nt <= 4));
}

WoSplitPlan wo_split_plan(int64_t M, int64_t N, int64_t K, int64_t ldx) {
  WoSplitPlan best;
  const Tuning& t = tuning();
  if (t.wo_split == 0 || M < 1 || M > 256 || (M + 64) * ldx * 2 >= kOutS || N * K >= kOutS || K % kStepK != 0) return best;
  // switches that force the other kernels' plans
  if (t.wo_split != 1 && (t.wo_stream || t.wo_plan_set || t.wo_msplit_set || t.wo_rows || t.wo_tile_min_w ||
                          t.wo_int8_tile2_min_m || t.wo_gemv_max_m >= 0 || t.wo_prefill_min_m != 65 || t.wo_prefill_s > 0 ||
                          t.wo_wide_mt >= 0 || t.wo_wide_s > 0 || t.wo_block == 1))
    return best;
  double bytes = 0.0;
  int64_t per_cu = 0;
  for (int mt = 1; mt <= 4; ++mt)
    for (int nt = 1; nt <= 5; ++nt) {
      const int64_t items = ((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * nt - 1) / (16 * nt)), cu = (items + 255) / 256;
      const double b = (double)cu * 16.0 * (2.0 * mt + nt) * (double)K;
      if (best.mt != 0 && b >= bytes) continue;
      best.mt = mt;
      best.nt = nt;
      bytes = b;
      per_cu = cu;
    }
  const int64_t steps = K / kStepK;
  best.nw = per_cu == 1 && steps >= 32 && best.nt <= (best.mt == 1 ? 3 : best.mt == 2 ? 2 : 0) ? 8 : 4;
  if (t.wo_split != 1 && !split_is_faster(best, per_cu, bytes, M, N, K)) best.mt = 0;
  return best;
}

int wo_split_launch(const WoSplitPlan& pl, const uint16_t* x, int64_t ldx, const uint8_t* w, const void* scale, int sd,
                    uint16_t* y, int64_t ldy, int64_t M, int N, int K, hipStream_t st, const char* name) {
  WoSplitParams p{};
  p.x = x;
  p.ldx = ldx;
  p.xbytes = (int)(((M - 1) * ldx + K) * 2);
  p.w = w;
  p.scale = scale;
  p.y = y;
  p.ldy = ldy;
  p.M = (int)M;
  p.N = N;
  p.K = K;
  p.vec_store = (reinterpret_cast<uintptr_t>(y) & 7) == 0 && ldy % 4 == 0;
  p.tiles_m = (int)((M + 16 * pl.mt - 1) / (16 * pl.mt));
  p.items = p.tiles_m * ((N + 16 * pl.nt - 1) / (16 * pl.nt));
#define MIQ_WS(MT_, NT_, NW_)                             \
  if (pl.mt == MT_ && pl.nt == NT_ && pl.nw == NW_) {     \
    go<MT_, NT_, NW_>(p, sd, st);                         \
    return check_launch(name);                            \
  }
#define MIQ_WS_MT(NT_) MIQ_WS(1, NT_, 4) MIQ_WS(2, NT_, 4) MIQ_WS(3, NT_, 4) MIQ_WS(4, NT_, 4)
  MIQ_WS_MT(1) MIQ_WS_MT(2) MIQ_WS_MT(3) MIQ_WS_MT(4) MIQ_WS_MT(5)
  MIQ_WS(1, 1, 8) MIQ_WS(1, 2, 8) MIQ_WS(1, 3, 8) MIQ_WS(2, 1, 8) MIQ_WS(2, 2, 8)
#undef MIQ_WS_MT
#undef MIQ_WS
  set_error("%s: no split kernel of %d x %d tiles, %d wavefronts", name, pl.mt, pl.nt, pl.nw);
  return MIQ_ERR_INVALID;
}

}  // namespace miq
