// How the block kernel (gemm_block.h) takes a call: its block shape and what a workgroup does with a row's slices. Host code
// only, a function of the sizes and the device's compute units, so that it can be asked without launching anything.
#pragma once

#include <math.h>
#include <stdint.h>

#include "gemm_args.h"

namespace dro {
namespace block {

// What a workgroup does with the slices of its rows: there is one; their sums are added in registers; or it takes one of
// them (blockIdx.y) and leaves its sums in a.partial, as the slab kernel does, for slab_reduce_kernel.
enum Slices { kOne, kAdded, kPart };

// The block shapes and what they were measured to take (us for 64 K tiles when every compute unit has n of them:
// per_block * n + once; MI355X, K = 4096 / 11008, 65 .. 4096 rows): small blocks leave no unit idle, large ones read less.
// bf16 and one-byte weights under the BF16 math have no 128 x 256: it takes twice a 128 x 128 block's time (74 n + 8), and a
// product never has more than twice as many of the smaller.
struct Shape {
  int bm, bn;
  float per_block, once;
};
template <int F, int MATH>
constexpr int kShapes = MATH == LX_MATH_BF16 && F != LX_W_NVFP4 ? 3 : 4;
template <int F, int MATH>
constexpr Shape shape(int i) {
  constexpr Shape bf16_math[4] = {{64, 64, 11, 10}, {64, 128, 20, 8}, {128, 128, 37, 2}, {}};
  constexpr Shape nvfp4[4] = {{64, 64, 17, 2}, {64, 128, 27, 6}, {128, 128, 50, 1}, {128, 256, 82, 2}};
  constexpr Shape int8_math[4] = {{64, 64, 14, 24}, {64, 128, 24, 22}, {128, 128, 45, 8}, {128, 256, 80, 10}};
  constexpr Shape fp8_math[4] = {{64, 64, 15, 28}, {64, 128, 28, 30}, {128, 128, 62, 2}, {128, 256, 106, 40}};
  return MATH == LX_MATH_INT8 ? int8_math[i] : MATH == LX_MATH_FP8 ? fp8_math[i] : F == LX_W_NVFP4 ? nvfp4[i] : bf16_math[i];
}

// The wide block (block_wide.h) as a plan's shape: 128 x 256, one wavefront a SIMD, quantised weights. It takes per_stage us a
// stage of K and per_block us a block besides (its first loads, the sums' way out), and once; under the FP8 math the blocks that
// start together take `first` more a stage. Measured on 65 .. 4096 rows, N 1024 .. 16384, K 1024 .. 14336, whole calls by the blocks of
// 64 .. 128 x 64 .. 256 and wide: 14336 x 4096 at 4096 rows fp8 582 / 433 us, NVFP4 700 / 497, INT8 math 318 / 285, FP8 math 551 / 387. A
// unit holds one block at a time and a block is a long chain: products of few blocks or short rows stay with the smaller shapes (fp8
// 3206 x 11968 at 338 rows 78 / 180, NVFP4 7536 x 3712 at 340 rows 66 / 79). The FP8 math's line was where its estimate of 1.55 a
// stage put it and kept 14336 x 4096 at 4096 rows from the wide block; of 24 other calls that `first` moved all are ahead (3 .. 35 %:
// 5194 x 6464 at 3747 rows 286 / 279, 12608 x 3840 at 2471 339 / 221), calls of one block a unit stay (behind: 3352 x 4672 at 1635 83 / 89; ahead:
// 12070 x 5248 at 456 103 / 92).
constexpr int kWide = 16;
struct WideCost {
  float per_stage, per_block, once, first = 0;
};
template <int F, int MATH>
constexpr WideCost wide_cost() {
  return MATH == LX_MATH_INT8 ? WideCost{0.82f, 8.5f, 3} : MATH == LX_MATH_FP8 ? WideCost{1.35f, 10, 4, 0.2f} : F == LX_W_NVFP4 ? WideCost{1.65f, 10, 4} : WideCost{0.75f, 8, 4};
}

// What the wide block is estimated to take, in us; infinite where it does not apply (block scales are loaded four bytes at a time).
template <int F, int MATH>
float wide_us(const GemmArgs& a, int units) {
  if (F == LX_W_BF16 || (F == LX_W_NVFP4 && (a.scale_row_bytes % 4 != 0 || reinterpret_cast<uintptr_t>(a.scale) % 4 != 0))) return INFINITY;
  constexpr WideCost c = wide_cost<F, MATH>();
  const int stages = MATH == LX_MATH_BF16 ? a.steps : (a.steps + 1) / 2;
  const int64_t blocks = static_cast<int64_t>((a.M + 127) / 128) * ((a.N + 255) / 256);
  return ((blocks + units - 1) / units) * (c.per_stage * stages + c.per_block) + c.first * stages + c.once;
}

// mode: Slices, or -1 where the kernel does not apply. K tiles of a row and of a slice.
struct Plan {
  int mode, shape, tiles, slice_tiles;
};

// Blocks of shape `i` a unit takes one behind the other, for `slices` launches of the product's.
template <int F, int MATH>
int64_t turns(const GemmArgs& a, int i, int slices, int units) {
  const Shape s = shape<F, MATH>(i);
  return (static_cast<int64_t>((a.M + s.bm - 1) / s.bm) * ((a.N + s.bn - 1) / s.bn) * slices + units - 1) / units;
}

// The shape that is estimated to take least for `slices` launches of `tiles` K tiles a block, and that time.
template <int F, int MATH>
int best_shape(const GemmArgs& a, int tiles, int slices, int units, float* us) {
  int best = 0;
  for (int i = 0; i < kShapes<F, MATH>; ++i) {
    const Shape s = shape<F, MATH>(i);
    const float t = (s.per_block * turns<F, MATH>(a, i, slices, units) + s.once) * tiles * (1.0f / 64);
    if (i == 0 || t < *us) {
      best = i;
      *us = t;
    }
  }
  return best;
}

// most: how many slices' sums there is a buffer for (0: none; kMaxSplit at most).
template <int F, int MATH>
Plan plan(const GemmArgs& a, int units, int most) {
  constexpr bool kBytes = MATH != LX_MATH_BF16;
  // Load steps a K tile holds (NVFP4: two tiles a step).
  constexpr int kSteps = kBytes || F == LX_W_BF16 ? 2 : 1, kTilesPerStep = F == LX_W_NVFP4 ? 2 : 1;
  // Offsets inside a block are 32 bits; a slice is whole pairs of tiles.
  if (a.row_bytes * 256 >= (1ll << 31) || (!kBytes && a.xs.ld * 2 * 256 >= (1ll << 31)) || a.steps_per_wave % (2 * kSteps)) return {-1, 0, 0, 0};
  const int tiles = ((a.steps * kTilesPerStep + kSteps - 1) / kSteps + 1) / 2 * 2;
  const int slice_tiles = a.steps_per_wave * kTilesPerStep / kSteps, slices = (tiles + slice_tiles - 1) / slice_tiles;
  float us = 0.0f;
  int whole = best_shape<F, MATH>(a, tiles, 1, units, &us);
  if (const float wide = wide_us<F, MATH>(a, units); wide < us) {
    whole = kWide;
    us = wide;
  }
  // One slice a workgroup: a second launch, and every slice's sums written and read once more (4.5 us and about 4 TB/s).
  auto parts = [&](int cut, int cuts, int* part) {
    float t;
    *part = best_shape<F, MATH>(a, cut, cuts, units, &t);
    return t + 4.5f + 8e-6f * a.M * a.N * cuts / 4.0f;
  };
  Plan best = {MATH != LX_MATH_INT8 && slices > 1 ? kAdded : kOne, whole, tiles, slice_tiles};
  if (int part; slices > 1 && most >= slices) {
    if (const float t = parts(slice_tiles, slices, &part); t < us) {
      best = {kPart, part, tiles, slice_tiles};
      us = t;
    }
  }
  if constexpr (MATH == LX_MATH_INT8) {
    // int32 sums are the same however K is cut. Where the row's own slices are taken, fewer that are estimated to take less (1418 x 576 x
    // 13312 13 -> 4 slices, 57.1 -> 40.5 us; 437 x 2608 x 10016 10 -> 3, 54.6 -> 36.9; 515 x 592 x 2656 6 -> 4 18.7 -> 17.2: rows, N, K; more
    // slices lost where they were estimated ahead, 79 x 1328 x 2240 5 -> 9 11.6 / 12.7). Where a workgroup walks all of K it stays so unless
    // its block is a large one and slices are estimated at 0.85 of the time: 515 x 4096 x 11008 in three 59.7 -> 53.1, 418 x 5216 x 13344 82 -> 70; of 14
    // others that the estimate alone moved eight lost (66 x 5360 x 2464 12.4 / 16.7). Nor do a row's own slices make way for blocks of more turns: one of 128 x
    // 256 a unit is as good as two of 64 x 128 (44 calls estimated at 0.85 .. 0.99: 0.91 .. 1.06, 154 x 6263 x 7584 37.4 / 39.8); and for 128 x 128 only where
    // that is estimated at 0.94 (18 calls above that: 0.91 .. 1.11, 112 x 11455 x 8192 41.7 / 46.3). 600 calls in slices drawn
    // afterwards (65 .. 4096 rows, N 512 .. 32768, K 1024 .. 14336): 0.87 on average with the sums' wider stores, none above 1.03; fewer columns were not measured.
    const bool own = best.mode == kPart;
    if (a.N >= 512 && (own || best.shape == 2 || best.shape == 3)) {
      const int64_t most_turns = own ? turns<F, MATH>(a, best.shape, slices, units) : INT64_MAX;
      const float large_us = own && best.shape == 3 ? 0.94f * us : INFINITY;
      if (!own) us *= 0.85f;
      for (int s = 2; s <= (own ? slices - 1 : most) && s * 2 <= tiles; ++s) {
        const int cut = ((tiles + s - 1) / s + 1) / 2 * 2;
        const int cuts = (tiles + cut - 1) / cut;
        int part;
        if (const float t = parts(cut, cuts, &part); t < us && (part != 2 || t < large_us) && turns<F, MATH>(a, part, cuts, units) <= most_turns) {
          best = {kPart, part, tiles, cut};
          us = t;
        }
      }
    }
  }
  return best;
}

}  // namespace block
}  // namespace dro
