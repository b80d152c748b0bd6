// The kernels of moe_block.h, one source per format (moe_block_<format>.hip).
#pragma once

#include "moe_block.h"

namespace dro {
namespace block {

// A tile of MT * 32 activation rows by 256 weight rows; gate/up: sixteen gate rows, their sixteen up rows, the next sixteen ...,
// so that a wavefront's four tiles are two pairs and SwiGLU is its epilogue.
template <int F, int MT, bool GATE_UP, bool SPLIT>
__device__ __forceinline__ void expert_tile(const ExpertBlock& a, int e, int g0, int rows, int c0, void* lds) {
  using B = Block<F, LX_MATH_BF16, 2, 4, MT, 4, SPLIT, true>;
  const int64_t first = static_cast<int64_t>(e) * (GATE_UP ? 2 : 1) * a.cols;  // the expert's first row in the stack
  // The stack row of the block's weight row, relative to c0's; a row past the last stands for the last.
  auto weight_row = [&](int row) {
    if constexpr (GATE_UP) return static_cast<uint32_t>(min(c0 + (row >> 5) * 16 + (row & 15), a.cols - 1) - c0 + ((row >> 4) & 1) * a.cols);
    else return static_cast<uint32_t>(min(c0 + row, a.cols - 1) - c0);
  };
  B b;
  b.init(GATE_UP ? a.x : a.x + static_cast<int64_t>(g0) * a.K, a.w.data + (first + c0) * a.row_bytes, a.w.scale + (first + c0) * a.scale_row_bytes,
         a.row_bytes, a.K, lds,
         [&](int row) {
           const int at = min(row, rows - 1);
           return static_cast<uint32_t>(GATE_UP ? a.order[g0 + at] / a.top_k : at) * static_cast<uint32_t>(a.K * 2);
         },
         [&](int row) { return weight_row(row) * static_cast<uint32_t>(a.row_bytes); },
         [&](int row) { return weight_row(row) * static_cast<uint32_t>(a.scale_row_bytes); });
  const int g4 = 4 * ((threadIdx.x & (kWave - 1)) >> 4);
  b.run(0, a.tiles, a.slice, [&](int m, int tile, const f32x4(&sums)[4]) {
    if (m >= rows) return;
    const float xs = a.xs ? a.xs[GATE_UP ? a.order[g0 + m] / a.top_k : g0 + m] : 1.0f;
    if constexpr (GATE_UP) {
#pragma unroll
      for (int t = 0; t < 4; t += 2) {
        const int c = c0 + 16 * ((tile + t) >> 1) + g4;
        if (c >= a.cols) continue;  // cols is a multiple of eight: all four or none
        uint32_t h[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = stack_factor(F, a.w, e, first + c + r) * (xs * sums[t][r]);
          const float u = stack_factor(F, a.w, e, first + c + r + a.cols) * (xs * sums[t + 1][r]);
          h[r] = f32_to_bf16_bits(silu(g) * u);
        }
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + static_cast<int64_t>(g0 + m) * a.cols + c) = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int c = c0 + 16 * (tile + t) + g4;
        if (c >= a.cols) continue;
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = stack_factor(F, a.w, e, first + c + r) * (xs * sums[t][r]);
        *reinterpret_cast<f32x4*>(static_cast<float*>(a.out) + static_cast<int64_t>(g0 + m) * a.cols + c) = v;
      }
    }
  });
}

template <int F, bool GATE_UP, bool SPLIT>
__global__ void __launch_bounds__(8 * kWave) __attribute__((amdgpu_waves_per_eu(2))) expert_block_kernel(const ExpertBlock a) {
  extern __shared__ __align__(16) f32x4 lds4[];
  constexpr int kCols = GATE_UP ? 128 : 256;
  const int blocks = (a.cols + kCols - 1) / kCols, live = *a.n_tiles * blocks;
  if (static_cast<int>(blockIdx.x) >= live) return;
  // A tile's blocks follow each other on one die, and the tiles of an expert behind one another.
  const int at = die_order(blockIdx.x, live), tile = at / blocks, c0 = (at - tile * blocks) * kCols;
  const int e = a.tile_expert[tile], g0 = a.tile_begin[tile], rows = a.tile_rows[tile];
  switch ((rows + 31) / 32) {
    case 1: expert_tile<F, 1, GATE_UP, SPLIT>(a, e, g0, rows, c0, lds4); break;
    case 2: expert_tile<F, 2, GATE_UP, SPLIT>(a, e, g0, rows, c0, lds4); break;
    case 3: expert_tile<F, 3, GATE_UP, SPLIT>(a, e, g0, rows, c0, lds4); break;
    default: expert_tile<F, 4, GATE_UP, SPLIT>(a, e, g0, rows, c0, lds4); break;
  }
}

template <int F>
int launch_experts(const ExpertBlock& a, int max_tiles, hipStream_t stream) {
  auto go = [&](auto kernel, int cols) {
    allow_lds(reinterpret_cast<const void*>(kernel), 144 * 1024);
    const unsigned grid = static_cast<unsigned>(max_tiles) * ((a.cols + cols - 1) / cols);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(8 * kWave), (Block<F, LX_MATH_BF16, 2, 4, 4, 4, true>::kLdsBytes), stream, a);
    return status_of(hipGetLastError());
  };
  const bool split = a.slice < (Block<F, LX_MATH_BF16, 2, 4, 4, 4, true>::kStepHalves ? 2 * a.tiles : a.tiles);
  if (a.order) return split ? go(expert_block_kernel<F, true, true>, 128) : go(expert_block_kernel<F, true, false>, 128);
  return split ? go(expert_block_kernel<F, false, true>, 256) : go(expert_block_kernel<F, false, false>, 256);
}

}  // namespace block
}  // namespace dro
