// lx_gemm_w for more rows than a decode step has (a prompt), on block_mfma.h: one launch for all M rows.
#pragma once

#include "block_mfma.h"
#include "gemm_args.h"

namespace dro {
namespace block {

// What a workgroup does with the slices of its rows: there is one; their sums are added in registers; or it takes one of
// them (blockIdx.y) and leaves its sums in a.partial, as the slab kernel does, for slab_reduce_kernel.
enum Slices { kOne, kAdded, kPart };

template <int F, int MATH, int WM, int WN, int MT, int NT, int MODE>
__global__ void __launch_bounds__(WM* WN* kWave) __attribute__((amdgpu_waves_per_eu(2))) gemm_block_kernel(const GemmArgs a, int tiles, int slice_tiles) {
  using B = Block<F, MATH, WM, WN, MT, NT, MODE == kAdded>;
  extern __shared__ __align__(16) f32x4 lds4[];
  const int blocks_m = (a.M + B::BM - 1) / B::BM, blocks_n = (a.N + B::BN - 1) / B::BN;
  // Blocks go by bands of kBand blocks of activation rows, across a band first: the blocks a die holds at once are about
  // as many rows high as wide, which is the least they read between them.
  constexpr int kBand = 8;
  const int at = die_order(blockIdx.x, blocks_m * blocks_n);
  const int band = at / (kBand * blocks_n), high = min(kBand, blocks_m - band * kBand), in_band = at - band * kBand * blocks_n;
  const int bn = in_band / high, bm = band * kBand + in_band - bn * high;
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
  const bool wide = !a.bias && a.beta == 0.0f && a.ld_y % 4 == 0 && reinterpret_cast<uintptr_t>(a.y) % 16 == 0;
  const bool bias_f32 = a.bias && a.bias_dtype == LX_F32;
  b.run(0, tiles, B::kStepHalves ? 2 * slice_tiles : slice_tiles, [&](int m, int tile, const typename B::Acc(&sums)[NT]) {
    if (m >= rows) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = 16 * (tile + t) + g4;
      if (n >= cols) continue;
      float rf[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        rf[r] = row_factor(F, a.scale, a.global, n0 + min(n + r, cols - 1));
        if (B::kBytes) rf[r] *= a.xscale[m0 + m];
      }
      if (wide && n + 3 < cols) {
        // write_out without bias and beta, four columns at a time.
        f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = a.alpha * ((!B::kBytes && a.act_scale ? rf[r] * a.act_scale[m0 + m] : rf[r]) * static_cast<float>(sums[t][r]));
        const int64_t at_y = static_cast<int64_t>(m0 + m) * a.ld_y + n0 + n;
        if (a.y_dtype == LX_F32) {
          *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + at_y) = v;
        } else {
          const u32x2 p = {f32_to_bf16_bits(v[0]) | static_cast<uint32_t>(f32_to_bf16_bits(v[1])) << 16,
                           f32_to_bf16_bits(v[2]) | static_cast<uint32_t>(f32_to_bf16_bits(v[3])) << 16};
          *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + at_y) = p;
        }
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (n + r < cols) {
          const float bias = !a.bias ? 0.0f : bias_f32 ? static_cast<const float*>(a.bias)[n0 + n + r] : load_as_f32(a.bias, a.bias_dtype, n0 + n + r);
          write_out(a, m0 + m, n0 + n + r, static_cast<float>(sums[t][r]), rf[r], bias);
        }
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

// The block shapes and what they were measured to take (us for 64 K tiles when every compute unit has n of them:
// per_block * n + once; MI355X, K = 4096 / 11008, 65 .. 4096 rows): small blocks leave no unit idle, large ones read less.
struct Shape {
  int bm, bn;
  float per_block, once;
};
template <int F, int MATH>
constexpr Shape shape(int i) {
  constexpr Shape bf16_math[4] = {{64, 64, 11, 10}, {64, 128, 20, 8}, {128, 128, 37, 2}, {128, 256, 74, 8}};
  constexpr Shape nvfp4[4] = {{64, 64, 17, 2}, {64, 128, 27, 6}, {128, 128, 50, 1}, {128, 256, 82, 2}};
  constexpr Shape int8_math[4] = {{64, 64, 14, 24}, {64, 128, 24, 22}, {128, 128, 45, 8}, {128, 256, 80, 10}};
  constexpr Shape fp8_math[4] = {{64, 64, 15, 28}, {64, 128, 28, 30}, {128, 128, 62, 2}, {128, 256, 106, 40}};
  return MATH == LX_MATH_INT8 ? int8_math[i] : MATH == LX_MATH_FP8 ? fp8_math[i] : F == LX_W_NVFP4 ? nvfp4[i] : bf16_math[i];
}

// The shape that is estimated to take least for `slices` launches of `tiles` K tiles a block, and that time.
template <int F, int MATH>
int best_shape(const GemmArgs& a, int tiles, int slices, float* us) {
  int best = 0;
  for (int i = 0; i < 4; ++i) {
    const Shape s = shape<F, MATH>(i);
    const int64_t blocks = static_cast<int64_t>((a.M + s.bm - 1) / s.bm) * ((a.N + s.bn - 1) / s.bn) * slices;
    const int64_t a_unit = (blocks + compute_units() - 1) / compute_units();
    const float t = (s.per_block * a_unit + s.once) * tiles * (1.0f / 64);
    if (i == 0 || t < *us) {
      best = i;
      *us = t;
    }
  }
  return best;
}

template <int F, int MATH, int MODE>
int launch_shape(int i, const GemmArgs& a, int tiles, int slice_tiles, hipStream_t stream) {
  switch (i) {
    case 0: return launch_mode<F, MATH, 2, 2, 2, 2, MODE>(a, tiles, slice_tiles, stream);
    case 1: return launch_mode<F, MATH, 2, 2, 2, 4, MODE>(a, tiles, slice_tiles, stream);
    case 2: return launch_mode<F, MATH, 2, 4, 4, 2, MODE>(a, tiles, slice_tiles, stream);
    default: return launch_mode<F, MATH, 2, 4, 4, 4, MODE>(a, tiles, slice_tiles, stream);
  }
}

template <int F, int MATH>
bool launch_format(const GemmArgs& a, int* status, hipStream_t stream) {
  constexpr bool kBytes = MATH != LX_MATH_BF16;
  // Load steps a K tile holds (NVFP4: two tiles a step).
  constexpr int kSteps = kBytes || F == LX_W_BF16 ? 2 : 1, kTilesPerStep = F == LX_W_NVFP4 ? 2 : 1;
  // Offsets inside a block are 32 bits; a slice is whole pairs of tiles.
  if (a.row_bytes * 256 >= (1ll << 31) || (!kBytes && a.xs.ld * 2 * 256 >= (1ll << 31)) || a.steps_per_wave % (2 * kSteps)) return false;
  const int tiles = ((a.steps * kTilesPerStep + kSteps - 1) / kSteps + 1) / 2 * 2;
  const int slice_tiles = a.steps_per_wave * kTilesPerStep / kSteps, slices = (tiles + slice_tiles - 1) / slice_tiles;
  float us = 0.0f, us_part = 0.0f;
  const int whole = best_shape<F, MATH>(a, tiles, 1, &us);
  if (a.partial) {
    // One slice a workgroup: a second launch, and every slice's sums written and read once more (4.5 us and about 4 TB/s).
    const int part = best_shape<F, MATH>(a, slice_tiles, slices, &us_part);
    us_part += 4.5f + 8e-6f * a.M * a.N * slices / 4.0f;
    if (us_part >= us) return false;
    *status = launch_shape<F, MATH, kPart>(part, a, tiles, slice_tiles, stream);
    return true;
  }
  *status = MATH != LX_MATH_INT8 && slices > 1 ? launch_shape<F, MATH, MATH != LX_MATH_INT8 ? kAdded : kOne>(whole, a, tiles, slice_tiles, stream)
                                               : launch_shape<F, MATH, kOne>(whole, a, tiles, slice_tiles, stream);
  return true;
}

}  // namespace block
}  // namespace dro
