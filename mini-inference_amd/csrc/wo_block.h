// Host interface of the INT8 block GEMMs (wo_block.hip): long prefill linears and the expert
// GEMMs of a MoE layer over many tokens.
#pragma once
#include <cstdint>

#include <hip/hip_runtime.h>

namespace miq {

// rows row0 .. row0 + 32 blocks - 1 of the padded expert layout, at most kMoeTileRows of them
constexpr int kMoeTileRows = 160;
struct MoeTile {
  int expert, row0, blocks, pad;
};

struct MoeBlockArgs {
  const uint16_t* hidden;  // [T, H]
  int T, H, I, E, topk;
  const uint8_t* gu_q;     // [E, 2 I, H]
  const void* gu_s;
  const uint8_t* dn_q;     // [E, H, I]
  const void* dn_s;
  int sd;
  const void* topk_w;
  int w_dtype;
  const MoeTile* tiles;
  const int32_t* num_tiles;
  const int32_t* sorted_ids;  // [max_rows], experts padded to 32 rows with T * topk
  int64_t max_rows;
  uint16_t* hbuf;             // [max_rows, I]
  uint16_t* ypair;            // [T * topk, H]
};

struct WidePlan;

// Whether an INT8 prefill call runs in 256 x 256 blocks rather than as the wide plan `wide`.
bool wo_block_planned(int64_t M, int64_t N, int64_t K, int64_t ldx, const WidePlan& wide);
int wo_block_launch(const uint16_t* x, int64_t ldx, const uint8_t* w, const void* scale, int sd, uint16_t* y, int64_t ldy,
                    int64_t M, int N, int K, hipStream_t st, const char* name);
bool moe_block_fits(int64_t T, int64_t topk, int64_t E, int64_t H, int64_t I, int64_t max_rows);
int moe_block_launch(const MoeBlockArgs& a, hipStream_t st, const char* name);

}  // namespace miq
