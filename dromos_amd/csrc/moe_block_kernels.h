// The kernels of moe_block.h, one source per format (moe_block_<format>.hip).
#pragma once

#include "block_wide.h"
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

// The same tile by the wide block: up to 16 * MT activation rows by 256 weight rows.
template <int F, int MT, bool GATE_UP>
__device__ __forceinline__ void expert_wide_tile(const ExpertBlock& a, int e, int g0, int rows, int c0, void* lds) {
  using B = Wide<F, LX_MATH_BF16, MT, true>;
  const int64_t first = static_cast<int64_t>(e) * (GATE_UP ? 2 : 1) * a.cols;
  const int64_t left = (GATE_UP ? 2 : 1) * a.cols - c0;  // the expert's rows from c0's on
  auto weight_row = [&](int row) {
    if constexpr (GATE_UP) return static_cast<uint32_t>(min(c0 + (row >> 5) * 16 + (row & 15), a.cols - 1) - c0 + ((row >> 4) & 1) * a.cols);
    else return static_cast<uint32_t>(min(c0 + row, a.cols - 1) - c0);
  };
  auto token = [&](int m) { return GATE_UP ? a.order[g0 + m] / a.top_k : g0 + m; };
  B b;
  b.init(GATE_UP ? a.x : a.x + static_cast<int64_t>(g0) * a.K, static_cast<int64_t>(GATE_UP ? a.x_rows : rows) * a.K * 2, a.w.data + (first + c0) * a.row_bytes,
         left * a.row_bytes, a.w.scale + (first + c0) * a.scale_row_bytes, left * a.scale_row_bytes, a.row_bytes, a.K, lds,
         [&](int row) {
           const int at = min(row, rows - 1);
           return static_cast<uint32_t>(GATE_UP ? a.order[g0 + at] / a.top_k : at) * static_cast<uint32_t>(a.K * 2);
         },
         [&](int row) { return weight_row(row) * static_cast<uint32_t>(a.row_bytes); },
         [&](int row) { return weight_row(row) * static_cast<uint32_t>(a.scale_row_bytes); });
  b.run((a.K * 2 + B::kXRow - 1) / B::kXRow, a.slice / (B::kNv ? 2 : 1));
  // Rows lane and 64 + lane's factors, handed round by row; the lane's columns' factors. All here before the loops.
  float xs[2] = {1.0f, 1.0f};
  if (a.xs) {
#pragma unroll
    for (int h = 0; h < 2; ++h) xs[h] = a.xs[token(min(64 * h + b.lane, rows - 1))];
  }
  if constexpr (GATE_UP) {
    // Half a wavefront a row: a lane's four values of the row's 128.
    const int at = b.lane & 31, piece = (at >> 2) * 8 + (at & 3), c = c0 + (at >> 2) * 16 + (at & 3) * 4;
    float fg[4], fu[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      fg[r] = stack_factor(F, a.w, e, first + min(c + r, a.cols - 1));
      fu[r] = stack_factor(F, a.w, e, first + min(c + r, a.cols - 1) + a.cols);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) asm volatile("" ::"v"(fg[r]), "v"(fu[r]), "v"(xs[r & 1]));
    for (int m0 = 2 * b.wave; m0 < rows; m0 += 2 * B::kWaves) {
      const int m = m0 + (b.lane >> 5);
      const float lo = __shfl(xs[0], m & 63), hi = __shfl(xs[1], m & 63), s = m < 64 ? lo : hi;
      if (m >= rows || c >= a.cols) continue;  // cols is a multiple of eight: all four or none
      const f32x4 sg = b.sum(m, piece), su = b.sum(m, piece + 4);
      uint32_t h[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) h[r] = f32_to_bf16_bits(silu(fg[r] * (s * sg[r])) * (fu[r] * (s * su[r])));
      *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.out) + static_cast<int64_t>(g0 + m) * a.cols + c) = u32x2{h[0] | h[1] << 16, h[2] | h[3] << 16};
    }
  } else {
    const int c = c0 + 4 * b.lane;
    float f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = stack_factor(F, a.w, e, first + min(c + r, a.cols - 1));
    asm volatile("" ::"v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "v"(xs[0]), "v"(xs[1]));
    for (int m = b.wave; m < rows; m += B::kWaves) {
      // (One lane's value each time: lanes without columns take no part in a choice between two.)
      const uint32_t s0 = __builtin_amdgcn_readlane(__float_as_uint(xs[0]), m & 63), s1 = __builtin_amdgcn_readlane(__float_as_uint(xs[1]), m & 63);
      const float s = __uint_as_float(m < 64 ? s0 : s1);
      f32x4 v = b.sum(m, b.lane);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = f[r] * (s * v[r]);
      if (c < a.cols) *reinterpret_cast<f32x4*>(static_cast<float*>(a.out) + static_cast<int64_t>(g0 + m) * a.cols + c) = v;
    }
  }
}

template <int F, bool GATE_UP>
__global__ void __launch_bounds__(4 * kWave) __attribute__((amdgpu_waves_per_eu(1, 1))) expert_wide_kernel(const ExpertBlock a) {
  extern __shared__ __align__(16) f32x4 lds4[];
  constexpr int kCols = GATE_UP ? 128 : 256;
  const int blocks = (a.cols + kCols - 1) / kCols, live = *a.n_tiles * blocks;
  if (static_cast<int>(blockIdx.x) >= live) return;
  const int at = die_order(blockIdx.x, live), tile = at / blocks, c0 = (at - tile * blocks) * kCols;
  const int e = __builtin_amdgcn_readfirstlane(a.tile_expert[tile]), g0 = __builtin_amdgcn_readfirstlane(a.tile_begin[tile]),
            rows = __builtin_amdgcn_readfirstlane(a.tile_rows[tile]);
  switch ((rows + 31) / 32) {
    case 1: expert_wide_tile<F, 2, GATE_UP>(a, e, g0, rows, c0, lds4); break;
    case 2: expert_wide_tile<F, 4, GATE_UP>(a, e, g0, rows, c0, lds4); break;
    case 3: expert_wide_tile<F, 6, GATE_UP>(a, e, g0, rows, c0, lds4); break;
    default: expert_wide_tile<F, 8, GATE_UP>(a, e, g0, rows, c0, lds4); break;
  }
}

template <int F>
int launch_experts(const ExpertBlock& a, int max_tiles, hipStream_t stream) {
  auto go = [&](auto kernel, int threads, int lds, int cols) {
    allow_lds(reinterpret_cast<const void*>(kernel), lds);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(max_tiles) * ((a.cols + cols - 1) / cols)), dim3(threads), lds, stream, a);
    return status_of(hipGetLastError());
  };
  if constexpr (F != LX_W_BF16) {
    if (a.wide) {
      constexpr int kLds[4] = {Wide<F, LX_MATH_BF16, 2, true>::kLdsBytes, Wide<F, LX_MATH_BF16, 4, true>::kLdsBytes, Wide<F, LX_MATH_BF16, 6, true>::kLdsBytes,
                               Wide<F, LX_MATH_BF16, 8, true>::kLdsBytes};
      int lds = 0;
      for (int bytes : kLds) lds = bytes > lds ? bytes : lds;
      return a.order ? go(expert_wide_kernel<F, true>, 4 * kWave, lds, 128) : go(expert_wide_kernel<F, false>, 4 * kWave, lds, 256);
    }
  }
  if constexpr (F == LX_W_BF16 || F == LX_W_NVFP4) {  // (the other formats are always wide)
    using B = Block<F, LX_MATH_BF16, 2, 4, 4, 4, true>;
    const bool split = a.slice < (B::kStepHalves ? 2 * a.tiles : a.tiles);
    if (a.order) return split ? go(expert_block_kernel<F, true, true>, 8 * kWave, B::kLdsBytes, 128) : go(expert_block_kernel<F, true, false>, 8 * kWave, B::kLdsBytes, 128);
    return split ? go(expert_block_kernel<F, false, true>, 8 * kWave, B::kLdsBytes, 256) : go(expert_block_kernel<F, false, false>, 8 * kWave, B::kLdsBytes, 256);
  }
  return kNotSupported;
}

}  // namespace block
}  // namespace dro
