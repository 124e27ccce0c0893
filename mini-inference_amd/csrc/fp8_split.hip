// FP8 x FP8 -> bf16 GEMM for decode batches and short or narrow prefill, gfx950: the sizes
// whose large tiles (fp8_gemm.hip) would leave most CUs idle.
//
//   y[m, n] = bf16( (sum_k xq[m,k] * wq[n,k]) * x_scale[m] * w_scale[n] )
//
// A workgroup owns a tile of 16 MT activation rows x 16 NT weight rows and its NW wavefronts
// split K between them: each multiplies the whole tile over its own k-steps of 128, with every
// operand loaded straight from memory into registers (no LDS staging, no barrier in the K loop),
// D k-steps ahead; the wavefronts' fp32 tiles are then added in LDS in wavefront order. 16 rows
// by N = 6144, K = 2560 so become 192 workgroups of 8 wavefronts with two or three k-steps each,
// instead of 48 workgroups that walk all 20 k-steps one after another.
#include "fp8_split.h"
#include "miq_common.h"

namespace miq {
namespace {

constexpr int kStep = kFp8Step;  // k per MFMA step
constexpr int kOutF = kFp8Outside;

struct SplitParams {
  const uint8_t* x;
  const float* xs;
  const uint8_t* w;
  const float* ws;
  uint16_t* y;
  int64_t ldy;
  int M, N, K;
  int tiles_m, items;
  bool vec_store;  // y rows 8-byte aligned (4 outputs per store)
};

// v_mfma_scale_f32_16x16x128_f8f6f4 with e4m3 operands and no block scales: A = 16 weight rows,
// B = 16 activation rows; lane (g, r) ends with outputs n = 4 g .. 4 g + 3 of activation row r.
__device__ inline f32x4 mfma128(const uint4 (&a)[2], const uint4 (&b)[2], f32x4 c) {
  const i32x8 av = {(int)a[0].x, (int)a[0].y, (int)a[0].z, (int)a[0].w, (int)a[1].x, (int)a[1].y, (int)a[1].z, (int)a[1].w};
  const i32x8 bv = {(int)b[0].x, (int)b[0].y, (int)b[0].z, (int)b[0].w, (int)b[1].x, (int)b[1].y, (int)b[1].z, (int)b[1].w};
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av, bv, c, 0, 0, 0, 0, 0, 0);
}

// NT weight tiles, MT activation tiles, NW wavefronts; D: k-steps of loads in flight.
// ONE: one activation tile row in all (the weights are read once: non-temporal loads).
template <int MT, int NT, int NW, int D, bool ONE>
__global__ void __launch_bounds__(NW * 64)
fp8_split_kernel(SplitParams p) {
  __shared__ __align__(16) f32x4 red[NW][MT * NT][64];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // XCD x (= workgroup id % 8) takes a contiguous eighth of the items, activation tiles
  // fastest, so the workgroups that read one weight tile share an L2
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int item = (int)((int64_t)p.items * xcd / 8) + local;
  if (item >= (int)((int64_t)p.items * (xcd + 1) / 8)) return;
  const int tn = item / p.tiles_m, tm = item - tn * p.tiles_m;
  const int n0 = tn * 16 * NT, m0 = tm * 16 * MT;
  const int steps = p.K / kStep;
  const int s0 = steps * wv / NW, s1 = steps * (wv + 1) / NW;  // this wavefront's k-steps

  const __amdgpu_buffer_rsrc_t wrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.w), 0, p.N * p.K, 0x00020000);
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.x), 0, p.M * p.K, 0x00020000);
  // weights: load h covers rows 8 h .. 8 h + 7 of a tile as whole 128-byte lines, in address
  // order within each 64-byte half; lanes_to_mfma turns two loads into the MFMA layout (lane
  // (g, r): row r, 16-byte chunks g and 4 + g). Rows past N or M lie past the buffers (zeros).
  const int lrr = (lane >> 2) & 7, lcl = lane & 3, lc2 = lane >> 5;
  const int bp_addr = (32 * (r >> 3) + 4 * (r & 7) + g) * 4;
  int woff[NT][2], xoff[MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int n = n0 + 16 * t + 8 * h + lrr;
      woff[t][h] = n < p.N ? n * p.K + lc2 * 64 + lcl * 16 : kOutF;
    }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + 16 * i + r;
    xoff[i] = m < p.M ? m * p.K + 16 * g : kOutF;
  }
  uint4 wq[D][NT][2], xq[D][MT][2];
  auto request = [&](int d, int s) {
    const int keep = (s - s1) >> 31;  // all ones while s is one of this wavefront's steps
    const int ko = s * kStep;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int ok = keep & ((woff[t][h] - kOutF) >> 31);
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(wrs, ((woff[t][h] + ko) & ok) | (kOutF & ~ok), 0, ONE ? 2 : 0);
        wq[d][t][h] = *reinterpret_cast<const uint4*>(&v);
      }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int ok = keep & ((xoff[i] - kOutF) >> 31);
      const int off = ((xoff[i] + ko) & ok) | (kOutF & ~ok);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        // (the second half's offset is in the instruction: past-the-end rows stay past the end)
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 64 * h, 0);
        xq[d][i][h] = *reinterpret_cast<const uint4*>(&v);
      }
    }
  };
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int d = 0; d < D; ++d) request(d, s0 + d);
  for (int s = s0; s < s1; s += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s + d < s1) {  // uniform
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          uint4 wf[2];
          lanes_to_mfma(bp_addr, wq[d][t][0], wq[d][t][1], wf[0], wf[1]);
#pragma unroll
          for (int i = 0; i < MT; ++i) acc[t][i] = mfma128(wf, xq[d][i], acc[t][i]);
        }
        request(d, s + d + D);
      }
    }
  }
  // the sum over the wavefronts, in wavefront order; (tile, lane) pairs are shared out over the
  // workgroup's threads
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < MT; ++i) red[wv][t * MT + i][lane] = acc[t][i];
  __syncthreads();
  for (int e = tid; e < MT * NT * 64; e += NW * 64) {
    const int ti = e >> 6, l = e & 63;
    f32x4 s = red[0][ti][l];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += red[w][ti][l];
    const int t = ti / MT, i = ti - t * MT;
    const int m = m0 + 16 * i + (l & 15), n = n0 + 16 * t + 4 * (l >> 4);
    if (m >= p.M || n >= p.N) continue;
    const float sx = p.xs[m];
    uint16_t* dst = p.y + (int64_t)m * p.ldy + n;
    if (p.vec_store && n + 4 <= p.N) {
      uint32_t o[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) o[v] = f32_to_bf16(s[v] * sx * p.ws[n + v]);
      *reinterpret_cast<uint2*>(dst) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (n + v < p.N) dst[v] = f32_to_bf16(s[v] * sx * p.ws[n + v]);
    }
  }
}

template <int MT, int NT, int NW>
void go(const SplitParams& p, hipStream_t st) {
  // loads in flight per wavefront: about 80 registers of operands
  constexpr int D = MT + NT <= 2 ? 5 : MT + NT <= 3 ? 3 : 2;
  const unsigned grid = (unsigned)((p.items + 7) / 8 * 8 + 8);  // every XCD's share fits
  if (p.tiles_m == 1)
    hipLaunchKernelGGL((fp8_split_kernel<MT, NT, NW, D, true>), dim3(grid), dim3(NW * 64), 0, st, p);
  else
    hipLaunchKernelGGL((fp8_split_kernel<MT, NT, NW, D, false>), dim3(grid), dim3(NW * 64), 0, st, p);
}

}  // namespace

// Launches the planned tile; operands below 2 GiB, K a multiple of 128.
int fp8_split_launch(const Fp8SplitPlan& pl, const uint8_t* xq, const float* xs, const uint8_t* wq, const float* ws,
                     uint16_t* y, int64_t ldy, int64_t M, int64_t N, int64_t K, hipStream_t st) {
  SplitParams p{xq, xs, wq, ws, y, ldy, (int)M, (int)N, (int)K, 0, 0, false};
  p.vec_store = (reinterpret_cast<uintptr_t>(y) & 7) == 0 && ldy % 4 == 0;
  p.tiles_m = (int)((M + 16 * pl.mt - 1) / (16 * pl.mt));
  p.items = p.tiles_m * (int)((N + 16 * pl.nt - 1) / (16 * pl.nt));
#define MIQ_FP8_SPLIT(MT_, NT_)                \
  if (pl.mt == MT_ && pl.nt == NT_) {          \
    if (pl.nw == 8) go<MT_, NT_, 8>(p, st);    \
    else if (pl.nw == 4) go<MT_, NT_, 4>(p, st); \
    else go<MT_, NT_, 2>(p, st);               \
    return check_launch("fp8_gemm");           \
  }
  MIQ_FP8_SPLIT(1, 1)
  MIQ_FP8_SPLIT(1, 2)
  MIQ_FP8_SPLIT(2, 1)
  MIQ_FP8_SPLIT(2, 2)
  MIQ_FP8_SPLIT(2, 4)
  MIQ_FP8_SPLIT(4, 2)
  MIQ_FP8_SPLIT(4, 4)
#undef MIQ_FP8_SPLIT
  set_error("fp8_gemm: no split kernel of %d x %d tiles", pl.mt, pl.nt);
  return MIQ_ERR_INVALID;
}

}  // namespace miq
