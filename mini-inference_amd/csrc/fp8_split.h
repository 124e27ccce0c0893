// Host interface of the split-K FP8 GEMM (fp8_split.hip), used by miq_fp8_gemm.
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

#include "fp8_plan.h"

namespace miq {

int fp8_split_launch(const Fp8SplitPlan& pl, const uint8_t* xq, const float* xs, const uint8_t* wq, const float* ws,
                     uint16_t* y, int64_t ldy, int64_t M, int64_t N, int64_t K, hipStream_t st);

}  // namespace miq
