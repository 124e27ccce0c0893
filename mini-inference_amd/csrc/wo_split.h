// Host interface of the INT8 split kernel for decode batches (wo_split.hip).
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

namespace miq {

// 16 mt x 16 nt tiles, nw wavefronts per workgroup that split K (mt = 0: not this kernel).
struct WoSplitPlan {
  int mt = 0, nt = 0, nw = 0;
};

WoSplitPlan wo_split_plan(int64_t M, int64_t N, int64_t K, int64_t ldx);
int wo_split_launch(const WoSplitPlan& pl, const uint16_t* x, int64_t ldx, const uint8_t* w, const void* scale, int sd,
                    uint16_t* y, int64_t ldy, int64_t M, int N, int K, hipStream_t st, const char* name);

}  // namespace miq
