// What the matrix-core products' kernels take: the call's operands and the launch geometry the host worked out,
// and the epilogue they share (engine/cpu/gemm.cpp:21-34).
#pragma once

#include "common.h"
#include "tile_mfma.h"

namespace dro {

constexpr size_t kLdsMax = 160 * 1024;  // LDS a workgroup may take

struct XRows {
  const void* x;
  int dtype;
  int64_t ld;  // elements between rows
};

struct GemmArgs {
  XRows xs;
  const uint8_t* w;
  const uint8_t* scale;
  float global;
  const void* bias;
  int bias_dtype;
  void* y;
  int y_dtype;
  int64_t ld_y;
  int M, N, K;
  float alpha, beta;
  int chunks, steps, steps_per_wave, S;
  int64_t row_bytes, scale_row_bytes;
  int tiles_per_wg, x_vecs, x_row_vecs, x_pitch, x_iters;  // the LDS activation image (XL kernels)
  int x_phased;  // lean kernel with two slices a wavefront: the image holds half of K at a time
  int win;       // windowed kernel: load steps of every slice the image holds at a time (2, 4 or 8)
  int win_steps_shift, win_shift, row_shift;  // log2 of win, of the 16-byte pieces in a window, and in an image row
  const int8_t* xq;     // the INT8 math: quantised activations [M, K], rows K bytes apart
  const float* xscale;  // and their per-row scales
  const float* act_scale;  // BF16-math kernels on a quantised math's activation images: the rows' scales (else null)
  int pass_begin, pass_steps, pass_continues;  // slab kernel: the part of every slice this launch takes, and whether it goes on from `partial`
  void* partial;  // slab kernel with S > 1: the slices' partial tiles, [S][tile][16 rows][lane] x 4 words (f32, or i32 for the INT8 math)
  int walk_slices;  // walk kernel with partial tiles: the slices a workgroup walks; split over a workgroup's wavefronts: the slices a wavefront walks
  int tuned;        // the variant table's entry for the call, or -1
  int walk_split;   // walk kernel: the wavefronts of a workgroup take one tile between them (two or four of them)
};

// The epilogue's operation order (engine/cpu/gemm.cpp:21-34); rf is the row factor, b the bias (0 without one).
__device__ __forceinline__ void write_out(const GemmArgs& a, int m, int n, float sum, float rf, float b) {
  float t = (a.act_scale ? rf * a.act_scale[m] : rf) * sum;
  if (a.bias) t += b;
  float v = a.alpha * t;
  const int64_t at = m * a.ld_y + n;
  if (a.beta != 0.0f) v = a.beta * load_as_f32(a.y, a.y_dtype, at) + v;
  store_from_f32(a.y, a.y_dtype, at, v);
}

__device__ __forceinline__ void write_out(const GemmArgs& a, int wtype, int m, int n, float sum) {
  write_out(a, m, n, sum, row_factor(wtype, a.scale, a.global, n), a.bias ? load_as_f32(a.bias, a.bias_dtype, n) : 0.0f);
}

// Four columns can be written at a time.
__device__ __forceinline__ bool wide_stores(const GemmArgs& a) {
  return !a.bias && a.beta == 0.0f && a.ld_y % 4 == 0 && reinterpret_cast<uintptr_t>(a.y) % 16 == 0;
}

// Four outputs at y[at] without bias and beta: write_out four columns at a time (rf: the row factors).
template <class Acc>
__device__ __forceinline__ void write_four(const GemmArgs& a, int64_t at, const Acc& sums, const float (&rf)[4]) {
  f32x4 v;
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = a.alpha * (rf[r] * static_cast<float>(sums[r]));
  if (a.y_dtype == LX_F32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + at) = v;
  } else {
    const bf16x2 p[2] = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + at) = __builtin_bit_cast(u32x2, p);
  }
}

// Columns n .. n + 3 of row m (of the matrix), as far as they exist, one at a time.
template <class Acc>
__device__ __forceinline__ void write_each(const GemmArgs& a, int m, int n, const Acc& sums, const float (&rf)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (n + r < a.N) {
      float t = rf[r] * static_cast<float>(sums[r]);
      if (a.bias) t += a.bias_dtype == LX_F32 ? static_cast<const float*>(a.bias)[n + r] : load_as_f32(a.bias, a.bias_dtype, n + r);
      float v = a.alpha * t;
      const int64_t at = m * a.ld_y + n + r;
      if (a.beta != 0.0f) v = a.beta * load_as_f32(a.y, a.y_dtype, at) + v;
      store_from_f32(a.y, a.y_dtype, at, v);
    }
}

// gemm_walk_<format>.hip: the walk kernel (gemm_walk.h) for up to 64 bf16 activation rows with W tiles a workgroup
// (1, 2 or 4; with a.partial set, 4 or 8, and a workgroup walks a.walk_slices slices and leaves their sums there; with a.walk_split
// set, W = 2 or 4 wavefronts on one tile); false when it does not apply to the call (the caller then takes another kernel), otherwise *status holds
// the launch's status.
bool launch_walk_bf16(const GemmArgs& a, int W, int* status, hipStream_t stream);
bool launch_walk_int8(const GemmArgs& a, int W, int* status, hipStream_t stream);
bool launch_walk_fp8(const GemmArgs& a, int W, int* status, hipStream_t stream);
bool launch_walk_nvfp4(const GemmArgs& a, int W, int* status, hipStream_t stream);

// gemm_ring_<format>.hip: the ring kernel (gemm_ring.h) for up to 64 bf16 activation rows with `cols` (32 or 64) weight rows a workgroup;
// false when it does not apply, otherwise *status holds the launch's status.
bool launch_ring_bf16(const GemmArgs& a, int cols, int* status, hipStream_t stream);
bool launch_ring_int8(const GemmArgs& a, int cols, int* status, hipStream_t stream);
bool launch_ring_fp8(const GemmArgs& a, int cols, int* status, hipStream_t stream);
bool launch_ring_nvfp4(const GemmArgs& a, int cols, int* status, hipStream_t stream);
// The same of its form with loader wavefronts, for 9 .. 64 rows on NVFP4 weights in up to four slices. Returns the launch's status.
int launch_fed_nvfp4(const GemmArgs& a, hipStream_t stream);

// gemm_block_<format>.hip: the block kernel (gemm_block.h) for any number of bf16 activation rows, gemm_block_<format>_math.hip the
// same under the INT8 and FP8 maths, as the plan says (gemm_block_plan.h). Returns the launch's status.
namespace block {
struct Plan;
}
int launch_block_bf16(const GemmArgs& a, const block::Plan& p, hipStream_t stream);
int launch_block_int8(const GemmArgs& a, const block::Plan& p, hipStream_t stream);
int launch_block_fp8(const GemmArgs& a, const block::Plan& p, hipStream_t stream);
int launch_block_nvfp4(const GemmArgs& a, const block::Plan& p, hipStream_t stream);
int launch_block_int8_math(const GemmArgs& a, const block::Plan& p, hipStream_t stream);
int launch_block_fp8_math(const GemmArgs& a, const block::Plan& p, hipStream_t stream);

}  // namespace dro
