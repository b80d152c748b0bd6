// The routed experts' two products for many tokens (a prompt), on block_mfma.h: a workgroup takes up to 128 of an expert's
// rows and 256 of its weight rows. The sums are the grouped kernels' (moe_grouped.hip) to the bit.
#pragma once

#include "block_mfma.h"
#include "moe_common.h"

namespace dro {

constexpr int kBlockTokens = 128;  // activation rows a tile of the block kernels holds at most

// One stage: gate/up (order set: position -> pair, whose token's row of x is multiplied; out is bf16 [P, cols], `cols`
// gate rows followed by as many up rows an expert) or down (x is [P, K] by position; out is f32 [P, cols]).
struct ExpertBlock {
  const uint16_t* x;
  const float* xs;  // the rows' scales under a quantised math (by token; by position), else null
  const int* order;
  int top_k;
  Stack w;
  const int *tile_expert, *tile_begin, *tile_rows, *n_tiles;
  void* out;
  int K, cols;
  int64_t row_bytes, scale_row_bytes;
  int tiles, slice;  // K tiles, and what a slice is of them (block_mfma.h: Block::run)
  int x_rows;        // rows of x
  bool wide;         // by block_wide.h (whose stages are a tile each, two of NVFP4's)
};

// moe_block_<format>.hip. max_tiles bounds *n_tiles (which only the device knows).
int launch_expert_block_bf16(const ExpertBlock& a, int max_tiles, hipStream_t stream);
int launch_expert_block_int8(const ExpertBlock& a, int max_tiles, hipStream_t stream);
int launch_expert_block_fp8(const ExpertBlock& a, int max_tiles, hipStream_t stream);
int launch_expert_block_nvfp4(const ExpertBlock& a, int max_tiles, hipStream_t stream);

}  // namespace dro
