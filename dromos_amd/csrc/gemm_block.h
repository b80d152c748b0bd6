// lx_gemm_w for more rows than a decode step has (a prompt), on block_mfma.h: one launch for all M rows.
#pragma once

#include "block_mfma.h"
#include "gemm_block_plan.h"

namespace dro {
namespace block {

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

template <int F, int MATH, int MODE>
int launch_shape(const GemmArgs& a, const Plan& p, hipStream_t stream) {
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
