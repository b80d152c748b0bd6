// lx_gemm_w for more rows than a decode step has (a prompt), on block_mfma.h: one launch for all M rows.
#pragma once

#include "block_mfma.h"
#include "block_wide.h"
#include "gemm_block_plan.h"

namespace dro {
namespace block {

// Where blocks lie: by bands of kBand blocks of activation rows, across a band first, so that the blocks a die holds at once
// are about as many rows high as wide, which is the least they read between them.
__device__ __forceinline__ void block_of(int b, int blocks_m, int blocks_n, int* bm, int* bn) {
  constexpr int kBand = 8;
  const int at = die_order(b, blocks_m * blocks_n);
  const int band = at / (kBand * blocks_n), high = min(kBand, blocks_m - band * kBand), in_band = at - band * kBand * blocks_n;
  *bn = in_band / high;
  *bm = band * kBand + in_band - *bn * high;
}

// The activation row's factor: its scale under a quantised math.
template <bool BYTES>
__device__ __forceinline__ float row_scale(const GemmArgs& a, int m) {
  return BYTES ? a.xscale[m] : a.act_scale ? a.act_scale[m] : 1.0f;
}

template <int F, int MATH, int WM, int WN, int MT, int NT, int MODE>
__global__ void __launch_bounds__(WM* WN* kWave) __attribute__((amdgpu_waves_per_eu(2))) gemm_block_kernel(const GemmArgs a, int tiles, int slice_tiles) {
  using B = Block<F, MATH, WM, WN, MT, NT, MODE == kAdded>;
  extern __shared__ __align__(16) f32x4 lds4[];
  int bm, bn;
  block_of(blockIdx.x, (a.M + B::BM - 1) / B::BM, (a.N + B::BN - 1) / B::BN, &bm, &bn);
  const int m0 = bm * B::BM, n0 = bn * B::BN;
  const int rows = min(B::BM, a.M - m0), cols = min(B::BN, a.N - n0);
  constexpr int xe = B::kBytes ? 1 : 2;
  const int64_t ld = B::kBytes ? a.K : a.xs.ld;
  const char* const x = B::kBytes ? reinterpret_cast<const char*>(a.xq) : static_cast<const char*>(a.xs.x);
  B b;
  b.init(x + m0 * ld * xe, a.w + n0 * a.row_bytes, F == LX_W_NVFP4 ? a.scale + n0 * a.scale_row_bytes : a.scale, a.row_bytes, a.K, lds4,
         [&](int row) { return static_cast<uint32_t>(min(row, rows - 1)) * static_cast<uint32_t>(ld * xe); },
         [&](int row) { return static_cast<uint32_t>(min(row, cols - 1)) * static_cast<uint32_t>(a.row_bytes); },
         [&](int row) { return static_cast<uint32_t>(min(row, cols - 1)) * static_cast<uint32_t>(a.scale_row_bytes); });
  const int lane = threadIdx.x & (kWave - 1), g4 = 4 * (lane >> 4);
  if constexpr (MODE == kPart) {
    const int n_tiles = (a.N + kTileRows - 1) / kTileRows, mts = (a.M + 15) / 16;
    typename B::Acc* const part = static_cast<typename B::Acc*>(a.partial) + static_cast<int64_t>(blockIdx.y) * n_tiles * mts * kWave + lane;
    const int first = blockIdx.y * slice_tiles;
    b.run(first, min(slice_tiles, tiles - first), 0, [&](int m, int tile, const typename B::Acc(&sums)[NT]) {
      const int mt = (m0 + m) >> 4;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int nt = (n0 >> 4) + tile + t;
        if (mt < mts && nt < n_tiles) part[(static_cast<int64_t>(nt) * mts + mt) * kWave] = sums[t];
      }
    });
    return;
  }
  const bool wide = wide_stores(a);
  b.run(0, tiles, B::kStepHalves ? 2 * slice_tiles : slice_tiles, [&](int m, int tile, const typename B::Acc(&sums)[NT]) {
    if (m >= rows) return;
    const float xs = row_scale<B::kBytes>(a, m0 + m);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = 16 * (tile + t) + g4;
      if (n >= cols) continue;
      float rf[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) rf[r] = row_factor(F, a.scale, a.global, n0 + min(n + r, cols - 1)) * xs;
      if (wide && n + 3 < cols) write_four(a, (m0 + m) * a.ld_y + n0 + n, sums[t], rf);
      else write_each(a, m0 + m, n0 + n, sums[t], rf);
    }
  });
}

template <int F, int MATH, int WM, int WN, int MT, int NT, int MODE>
int launch_mode(const GemmArgs& a, int tiles, int slice_tiles, hipStream_t stream) {
  using B = Block<F, MATH, WM, WN, MT, NT, MODE == kAdded>;
  const auto kernel = gemm_block_kernel<F, MATH, WM, WN, MT, NT, MODE>;
  allow_lds(reinterpret_cast<const void*>(kernel), kLdsMax);
  const int64_t blocks = static_cast<int64_t>((a.M + B::BM - 1) / B::BM) * ((a.N + B::BN - 1) / B::BN);
  const int slices = MODE == kPart ? (tiles + slice_tiles - 1) / slice_tiles : 1;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks), slices), dim3(B::kThreads), B::kLdsBytes, stream, a, tiles, slice_tiles);
  return status_of(hipGetLastError());
}

// The wide block (block_wide.h): 128 x 256, all of K in a workgroup.
template <int F, int MATH, int MODE>
__global__ void __launch_bounds__(4 * kWave) __attribute__((amdgpu_waves_per_eu(1, 1))) gemm_wide_kernel(const GemmArgs a, int stages, int slice) {
  using B = Wide<F, MATH, 8, MODE == kAdded>;
  extern __shared__ __align__(16) f32x4 lds4[];
  int bm, bn;
  block_of(blockIdx.x, (a.M + B::BM - 1) / B::BM, (a.N + B::BN - 1) / B::BN, &bm, &bn);
  const int m0 = bm * B::BM, n0 = bn * B::BN;
  const int rows = min(B::BM, a.M - m0), cols = min(B::BN, a.N - n0);
  constexpr int xe = B::kBytes ? 1 : 2;
  const int64_t ld = (B::kBytes ? a.K : a.xs.ld) * xe;
  const char* const x = B::kBytes ? reinterpret_cast<const char*>(a.xq) : static_cast<const char*>(a.xs.x);
  B b;
  b.init(x + m0 * ld, (rows - 1) * ld + a.K * xe, a.w + n0 * a.row_bytes, cols * a.row_bytes, F == LX_W_NVFP4 ? a.scale + n0 * a.scale_row_bytes : a.scale,
         cols * a.scale_row_bytes, a.row_bytes, a.K, lds4, [&](int row) { return static_cast<uint32_t>(min(row, rows - 1)) * static_cast<uint32_t>(ld); },
         [&](int row) { return static_cast<uint32_t>(min(row, cols - 1)) * static_cast<uint32_t>(a.row_bytes); },
         [&](int row) { return static_cast<uint32_t>(min(row, cols - 1)) * static_cast<uint32_t>(a.scale_row_bytes); });
  const bool wide = wide_stores(a);
  b.run(stages, slice);
  // A wavefront writes every fourth row, a lane its four columns. What comes from memory is asked for in front of the loop (a load in
  // it would wait behind the stores: 700 cycles a row).
  const int n = 4 * b.lane;
  float rf[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) rf[r] = row_factor(F, a.scale, a.global, n0 + min(n + r, cols - 1));
  float xs[2];  // rows lane and 64 + lane
#pragma unroll
  for (int h = 0; h < 2; ++h) xs[h] = row_scale<B::kBytes>(a, m0 + min(64 * h + b.lane, rows - 1));
  // (Everything is here: no wait in the loops, where it would be one for the stores too.)
  asm volatile("" ::"v"(rf[0]), "v"(rf[1]), "v"(rf[2]), "v"(rf[3]), "v"(xs[0]), "v"(xs[1]));
  // (One lane's value each time, and the loops are walked by every lane: a value taken from a lane that is switched off would be
  // whatever the register allocation left there. Lanes without columns only do not store.)
  auto factors = [&](int m, float(&f)[4]) {
    const uint32_t s0 = __builtin_amdgcn_readlane(__float_as_uint(xs[0]), m & 63), s1 = __builtin_amdgcn_readlane(__float_as_uint(xs[1]), m & 63);
    const float s = __uint_as_float(m < 64 ? s0 : s1);
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = rf[r] * s;
  };
  float f[4];
  if (wide && cols % 4 == 0) {
    for (int m = b.wave; m < rows; m += B::kWaves) {
      factors(m, f);
      const typename B::Acc sums = b.sum(m, b.lane);
      if (n < cols) write_four(a, (m0 + m) * a.ld_y + n0 + n, sums, f);
    }
  } else {
    for (int m = b.wave; m < rows; m += B::kWaves) {
      factors(m, f);
      const typename B::Acc sums = b.sum(m, b.lane);
      if (wide && n + 3 < cols) write_four(a, (m0 + m) * a.ld_y + n0 + n, sums, f);
      else if (n < cols) write_each(a, m0 + m, n0 + n, sums, f);
    }
  }
}

template <int F, int MATH, int MODE>
int launch_wide(const GemmArgs& a, const Plan& p, hipStream_t stream) {
  using B = Wide<F, MATH, 8, MODE == kAdded>;
  const auto kernel = gemm_wide_kernel<F, MATH, MODE>;
  allow_lds(reinterpret_cast<const void*>(kernel), kLdsMax);
  const int64_t blocks = static_cast<int64_t>((a.M + B::BM - 1) / B::BM) * ((a.N + B::BN - 1) / B::BN);
  constexpr int kSteps = B::kBytes ? 2 : 1;  // load steps a stage
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(B::kThreads), B::kLdsBytes, stream, a, (a.steps + kSteps - 1) / kSteps, a.steps_per_wave / kSteps);
  return status_of(hipGetLastError());
}

template <int F, int MATH, int MODE>
int launch_shape(const GemmArgs& a, const Plan& p, hipStream_t stream) {
  if constexpr (F != LX_W_BF16 && MODE != kPart)
    if (p.shape == kWide) return launch_wide<F, MATH, MODE>(a, p, stream);
  switch (p.shape) {
    case 0: return launch_mode<F, MATH, 2, 2, 2, 2, MODE>(a, p.tiles, p.slice_tiles, stream);
    case 1: return launch_mode<F, MATH, 2, 2, 2, 4, MODE>(a, p.tiles, p.slice_tiles, stream);
    case 2: return launch_mode<F, MATH, 2, 4, 4, 2, MODE>(a, p.tiles, p.slice_tiles, stream);
    default:
      if constexpr (kShapes<F, MATH> > 3) return launch_mode<F, MATH, 2, 4, 4, 4, MODE>(a, p.tiles, p.slice_tiles, stream);
      else return kNotSupported;
  }
}

template <int F, int MATH>
int launch_format(const GemmArgs& a, const Plan& p, hipStream_t stream) {
  if (p.mode == kPart) return launch_shape<F, MATH, kPart>(a, p, stream);
  if constexpr (MATH != LX_MATH_INT8)  // (int32 sums need no slices)
    if (p.mode == kAdded) return launch_shape<F, MATH, kAdded>(a, p, stream);
  return launch_shape<F, MATH, kOne>(a, p, stream);
}

}  // namespace block
}  // namespace dro
