// Host interface of the split-K FP8 GEMM (fp8_split.hip), used by miq_fp8_gemm.
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

namespace miq {

// 16 mt x 16 nt tiles, nw wavefronts per workgroup that split K, and the modelled time.
struct Fp8SplitPlan {
  int mt = 0, nt = 0, nw = 0;
  double us = 0.0;
};

Fp8SplitPlan fp8_split_plan(int64_t M, int64_t N, int64_t K);
int fp8_split_launch(const Fp8SplitPlan& pl, const uint8_t* xq, const float* xs, const uint8_t* wq, const float* ws,
                     uint16_t* y, int64_t ldy, int64_t M, int64_t N, int64_t K, hipStream_t st);

}  // namespace miq
