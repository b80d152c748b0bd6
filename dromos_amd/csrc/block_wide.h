// The product of many activation rows by quantised weights with one wavefront a SIMD: 16 * MT activation rows by 256 weight
// rows, every wavefront all of the activation rows by 64 weight rows of its own. The sums are block_mfma.h's to the bit (the
// same instruction on the same k in the same order, the same slices).
//
// Against block_mfma.h's blocks: a weight is expanded to bf16 by the one wavefront that uses it and never lies expanded in LDS,
// and an activation fragment read from LDS meets four weight tiles instead of two. A compute unit has registers for the two sets
// of sums (a slice's, and the slices' before it) of 128 x 256 values and what is left of them is worth more as one wavefront's:
// 128 x 64 sums a wavefront take half of the LDS reads that 64 x 64 take.
//
// Both operands go from memory straight into LDS (buffer loads with an LDS destination), a ring of stages deep, as they lie in
// memory: no staging registers, no address arithmetic in the walk. A stage is one load step: 64 bytes of a weight row (two under
// the byte maths) and the activations against them. In LDS a row's pieces of 16 bytes are turned by the row (piece ^ row) so that
// the lanes of a fragment read that are served together fall into different banks.
#pragma once

#include "common.h"
#include "tile_mfma.h"

namespace dro {
namespace block {

using Rsrc = __attribute__((ext_vector_type(4))) int32_t;

// A buffer of `bytes` bytes: no load reaches past it.
__device__ __forceinline__ Rsrc buffer_of(const void* base, int64_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return Rsrc{__builtin_amdgcn_readfirstlane(static_cast<int>(p)), __builtin_amdgcn_readfirstlane(static_cast<int>(p >> 32) & 0xffff),
              __builtin_amdgcn_readfirstlane(static_cast<int>(bytes)), 0x00020000};
}

// 16 (4) bytes a lane from buffer + voffset + soffset to LDS address `lds` + 16 (4) * lane. Counted by vmcnt; the compiler does not
// know of them (it would wait for all of them before any LDS read), so wait_loads() does. (M0 is reserved: the compiler keeps nothing in it.)
__device__ __forceinline__ void load_to_lds16(uint32_t lds, uint32_t voffset, const Rsrc& rsrc, uint32_t soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}
__device__ __forceinline__ void load_to_lds4(uint32_t lds, uint32_t voffset, const Rsrc& rsrc, uint32_t soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(voffset), "s"(rsrc), "s"(soffset) : "memory");
}

// Waits until at most LEFT of this wavefront's loads are on their way and all of its LDS reads and writes are done.
template <int LEFT>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
}

// Values 2 p and 2 p + 1 of instruction j's eight (tile_mfma.h: weight_fragment) as two bf16.
template <int F>
__device__ __forceinline__ uint32_t weight_pair(const u32x4& w, uint32_t scales, int j, int p) {
  if constexpr (F == LX_W_NVFP4) {
    const uint32_t d = w[j];
    const float s = j < 2 ? e4m3_byte_to_f32<0>(scales) : e4m3_byte_to_f32<1>(scales);
    const f32x2 v = p == 0   ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 0)
                    : p == 1 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 1)
                    : p == 2 ? __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 2)
                             : __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(d, 1.0f, 3);
    return __builtin_bit_cast(uint32_t, pack_bf16(v.x * s, v.y * s));
  } else {
    const uint32_t d = w[2 * j + (p >> 1)];
    if constexpr (F == LX_W_FP8) {
      return __builtin_bit_cast(uint32_t, p & 1 ? __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, true) : __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, 1.0f, false));
    } else {
      const int at = 16 * (p & 1);
      return __builtin_bit_cast(uint32_t, pack_bf16(static_cast<float>(static_cast<int>(static_cast<int8_t>(d >> at))), static_cast<float>(static_cast<int>(static_cast<int8_t>(d >> (at + 8))))));
    }
  }
}

template <int F, int MATH, int MT, bool SPLIT>
struct Wide {
  static_assert(F != LX_W_BF16, "quantised weights");
  static constexpr bool kBytes = MATH != LX_MATH_BF16;  // one-byte operands on both sides
  static constexpr bool kNv = F == LX_W_NVFP4;
  static constexpr int kWaves = 4, kThreads = kWaves * kWave;
  static constexpr int NT = 4;                // tiles of weight rows a wavefront
  static constexpr int BM = MT * 16, BN = kWaves * NT * 16;
  static constexpr int J = kNv ? 4 : 2;       // matrix instructions (k) a stage
  static constexpr int kXRow = kNv ? 256 : 128, kWRow = kBytes ? 128 : 64;  // bytes of a row a stage
  // Wave-sized loads a stage, per wavefront; a region is a whole number of them for all four.
  static constexpr int kXLoads = (BM * kXRow + 4095) / 4096, kWLoads = BN * kWRow / 4096, kSLoads = kNv ? 2 : 0;
  static constexpr int kLoads = kXLoads + kWLoads + kSLoads;
  static constexpr int kWAt = kXLoads * 4096, kSAt = kWAt + kWLoads * 4096, kStage = kSAt + kSLoads * 1024;
  static constexpr int kStages = 160 * 1024 / kStage < 5 ? 160 * 1024 / kStage : 5;
  static constexpr int kLdsBytes = kStages * kStage;
  static_assert(BM * 1024 <= kLdsBytes, "room for the block's sums");
  static_assert(kStages >= 3, "a ring of three stages at least");
  using Acc = typename std::conditional<MATH == LX_MATH_INT8, i32x4, f32x4>::type;

  Rsrc xbuf, wbuf, sbuf;
  uint32_t xrow[kXLoads], wrow[kWLoads], srow[kSLoads > 0 ? kSLoads : 1];  // this lane's 16 (4) bytes of every load
  int xpiece, wpiece, spiece;  // and their place in the stage's row
  int K, xbytes, wbytes;       // a row's bytes
  uint8_t* lds;
  uint32_t lds_at;
  int lane, wave, g, i;

  // xoff(row) / woff(row) / soff(row): byte offsets of activation row / weight row / weight row's scales from the bases, for rows
  // of this block (the caller clamps to rows that exist); xsize / wsize / ssize: bytes from the bases that may be read.
  template <class XOff, class WOff, class SOff>
  __device__ __forceinline__ void init(const void* xb, int64_t xsize, const void* wb, int64_t wsize, const void* sb, int64_t ssize, int64_t row_bytes, int K_, void* lds_,
                                       XOff xoff, WOff woff, SOff soff) {
    lane = threadIdx.x & (kWave - 1);
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    g = lane >> 4;
    i = lane & 15;
    K = K_;
    xbytes = kBytes ? K : K * 2;
    wbytes = static_cast<int>(row_bytes);
    lds = static_cast<uint8_t*>(lds_);
    lds_at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds)));
    xbuf = buffer_of(xb, xsize);
    wbuf = buffer_of(wb, wsize);
    sbuf = buffer_of(sb, ssize);
    {
      // Rows of kXRow bytes: place p of a row is for instruction p / 4's lanes of group p % 4; slot s of row r holds place s ^ r.
      constexpr int kSlots = kXRow / 16;
#pragma unroll
      for (int u = 0; u < kXLoads; ++u) {
        const int at = (u * kWaves + wave) * kWave + lane, row = at / kSlots, place = (at ^ row) % kSlots;
        xpiece = (kBytes ? place : J * (place & 3) + (place >> 2)) * 16;
        xrow[u] = xoff(min(row, BM - 1)) + static_cast<uint32_t>(xpiece);
      }
    }
    {
      // Weight rows of 64 bytes: slot s holds piece s ^ (r / 2 % 4); of 128 as the activations.
      constexpr int kSlots = kWRow / 16;
#pragma unroll
      for (int u = 0; u < kWLoads; ++u) {
        const int at = (u * kWaves + wave) * kWave + lane, row = at / kSlots;
        wpiece = ((at % kSlots) ^ (kBytes ? row & 7 : (row >> 1) & 3)) * 16;
        wrow[u] = woff(row) + static_cast<uint32_t>(wpiece);
      }
    }
    spiece = (lane & 1) * 4;
#pragma unroll
    for (int u = 0; u < kSLoads; ++u) srow[u] = soff((u * kWaves + wave) * 32 + (lane >> 1)) + static_cast<uint32_t>(spiece);
  }

  // Asks for load u of stage st into ring slot `slot`: weights first. What lies past a row's end is asked for at its start instead
  // (and zeroed by finish()).
  __device__ __forceinline__ void load(int st, int slot, int u) const {
    const uint32_t to = lds_at + slot * kStage;
    if (u < kWLoads) {
      const uint32_t back = wpiece + st * kWRow >= wbytes ? wpiece : 0;
      load_to_lds16(to + kWAt + wave * 1024 + u * 4096, wrow[u] - back, wbuf, st * kWRow);
    } else if (u < kWLoads + kSLoads) {
      const uint32_t back = spiece + st * 8 >= K / 16 ? spiece : 0;
      load_to_lds4(to + kSAt + wave * 256 + (u - kWLoads) * 1024, srow[u - kWLoads] - back, sbuf, st * 8);
    } else {
      const uint32_t back = xpiece + st * kXRow >= xbytes ? xpiece : 0;
      load_to_lds16(to + wave * 1024 + (u - kWLoads - kSLoads) * 4096, xrow[u - kWLoads - kSLoads] - back, xbuf, st * kXRow);
    }
  }

  // Stage st, which reaches past the row's end, once this wavefront's loads of it have arrived: zeros there, on both sides (a
  // weight's code there could be a NaN).
  __device__ __forceinline__ void finish(int st, int slot) const {
    uint8_t* const to = lds + slot * kStage;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    if (xpiece + st * kXRow >= xbytes) {
#pragma unroll
      for (int u = 0; u < kXLoads; ++u) *reinterpret_cast<u32x4*>(to + u * 4096 + wave * 1024 + lane * 16) = zero;
    }
    if (wpiece + st * kWRow >= wbytes) {
#pragma unroll
      for (int u = 0; u < kWLoads; ++u) *reinterpret_cast<u32x4*>(to + kWAt + u * 4096 + wave * 1024 + lane * 16) = zero;
    }
    if constexpr (kNv) {
#pragma unroll
      for (int u = 0; u < kSLoads; ++u) {
        uint8_t* const s = to + kSAt + u * 1024 + wave * 256 + lane * 4;
        if (spiece + st * 8 >= K / 16) *reinterpret_cast<uint32_t*>(s) = 0;
        else if (spiece + st * 8 + 2 >= K / 16) *reinterpret_cast<uint16_t*>(s + 2) = 0;
      }
    }
  }

  // The products of `stages` stages in slices of `slice`; behind it the sums lie in LDS for sum() to read.
  __device__ __forceinline__ void run(int stages, int slice) {
    // Where a stage's fragments are read.
    uint32_t xat[J];
#pragma unroll
    for (int j = 0; j < J; ++j) xat[j] = i * kXRow + ((4 * j + g) ^ (i % (kXRow / 16))) * 16;
    const uint32_t wat0 = kWAt + (wave * 64 + i) * kWRow + (kBytes ? g ^ (i & 7) : g ^ ((i >> 1) & 3)) * 16;
    const uint32_t wat1 = kBytes ? wat0 ^ 64 : wat0;
    const uint32_t sat = kSAt + (wave * 64 + i) * 8 + g * 2;
    const bool cut = stages * kXRow > xbytes;  // the last stage reaches past the row
    Acc acc[NT][MT], tot[SPLIT ? NT : 1][SPLIT ? MT : 1];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[nt][mt] = Acc{0, 0, 0, 0};
        if constexpr (SPLIT) tot[nt][mt] = Acc{0, 0, 0, 0};
      }
    u32x4 raw[NT];
    uint32_t sc[NT];
    u32x4 wf[2][NT], xf[2][MT];
    auto fetch_raw = [&](const uint8_t* st, int nt) {
      if constexpr (!kBytes) raw[nt] = *reinterpret_cast<const u32x4*>(st + wat0 + nt * 16 * kWRow);
      sc[nt] = 0;
      if constexpr (kNv) sc[nt] = *reinterpret_cast<const uint16_t*>(st + sat + nt * 128);
    };
    // Part p (of four) of fragment nt of instruction j: two values of a lane's eight.
    auto fetch_w = [&](u32x4(&w)[NT], const uint8_t* st, int j, int nt, int p) {
      if constexpr (!kBytes) w[nt][p] = weight_pair<F>(raw[nt], sc[nt], j, p);
      else if (p == 0) w[nt] = *reinterpret_cast<const u32x4*>(st + (j & 1 ? wat1 : wat0) + nt * 16 * kWRow);
    };
    auto fetch_x = [&](u32x4(&x)[MT], const uint8_t* st, int j, int mt) {
      x[mt] = *reinterpret_cast<const u32x4*>(st + xat[j] + mt * 16 * kXRow);
    };
#pragma unroll
    for (int st = 0; st < kStages - 1; ++st)
      if (st < stages) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) load(st, st, u);
      }
    // Before anyone reads stage st: this wavefront's loads of it are here (those of the stages behind it, kStages - 2 at most, may be
    // on their way), and behind the barrier everyone's are.
    auto arrive = [&](auto steady, int st, int slot) {
      const int behind = min(stages - 1 - st, kStages - 2);
      if (decltype(steady)::value || behind == kStages - 2) wait_loads<(kStages - 2) * kLoads>();
      else if (kStages > 4 && behind == kStages - 3) wait_loads<(kStages > 4 ? kStages - 3 : 0) * kLoads>();
      else if (kStages > 3 && behind == 1) wait_loads<kLoads>();
      else wait_loads<0>();
      if (!decltype(steady)::value && cut && st == stages - 1) {
        finish(st, slot);
        wait_loads<0>();
      }
      asm volatile("s_barrier" ::: "memory");
    };
    arrive(std::false_type{}, 0, 0);
    if (kStages - 1 < stages) {
#pragma unroll
      for (int u = 0; u < kLoads; ++u) load(kStages - 1, kStages - 1, u);
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      fetch_raw(lds, nt);
#pragma unroll
      for (int p = 0; p < 4; ++p) fetch_w(wf[0], lds, 0, nt, p);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) fetch_x(xf[0], lds, 0, mt);
    int slot = 0;
    // Stage st. Under instruction j's products the next one's fragments are read and expanded; the last one's next are the next
    // stage's. Behind the barrier in front of the last one's products nobody reads this stage any more: its slot takes the stage
    // kStages further on. The order is written down group by group (a group: an activation tile's products), because the wavefront
    // is alone on its SIMD: every instruction between two products is free as long as there are no more than three (the matrix cores
    // take 16 cycles a product, an instruction is issued every four), and a read that is used at once stops everything.
    auto step = [&](auto steady, int st) {
      const int next = slot + 1 == kStages ? 0 : slot + 1;
      const uint8_t *const here = lds + slot * kStage, *const there = lds + next * kStage;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const bool last = j == J - 1;
        const uint8_t* const from = last ? there : here;
        __builtin_amdgcn_sched_barrier(0);
        if (last) arrive(steady, st + 1, next);
        // Where the next weights are expanded: behind their read's latency if it is the next stage's.
        const int first = last ? (MT + 2) / 4 : 0;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          if (last && mt == 0) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) fetch_raw(from, nt);
          }
#pragma unroll
          for (int r = 0; r < MT; ++r)
            if (r / 2 == mt) fetch_x(xf[(j + 1) & 1], from, (j + 1) % J, r);
#pragma unroll
          for (int d = 0; d < NT * 4; ++d)
            if (first + d * (MT - first) / (NT * 4) == mt) fetch_w(wf[(j + 1) & 1], from, (j + 1) % J, d / 4, d % 4);
          if (decltype(steady)::value && last) {
#pragma unroll
            for (int u = 0; u < kLoads; ++u)
              if (u * MT / kLoads == mt) load(st + kStages, slot, u);
          }
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            if constexpr (kBytes) acc[nt][mt] = byte_mfma<MATH>(__builtin_bit_cast(i32x4, wf[j & 1][nt]), __builtin_bit_cast(i32x4, xf[j & 1][mt]), acc[nt][mt]);
            else acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[j & 1][nt]), __builtin_bit_cast(bf16x8, xf[j & 1][mt]), acc[nt][mt], 0, 0, 0);
          }
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, kNv ? 3 : 2, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      slot = next;
    };
    for (int st = 0, end = SPLIT ? slice : stages;; end += slice) {
      for (const int full = min(end, stages - kStages); st < full; ++st) step(std::true_type{}, st);
      for (const int all = min(end, stages); st < all; ++st) step(std::false_type{}, st);
      if (!SPLIT || st >= stages) break;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          tot[nt][mt] += acc[nt][mt];
          acc[nt][mt] = Acc{0, 0, 0, 0};
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    // The sums go through LDS, a row's 256 (1 KB) together, its pieces of four turned by the row, so that whole rows are written out
    // by a short loop: written from where the products leave them, a wavefront alone on its SIMD walked 32 pieces of unrolled code
    // once each and waited for the row factors and for the code itself, 20 us a block.
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        Acc sums = acc[nt][mt];
        if constexpr (SPLIT) sums = tot[nt][mt] + sums;
        *reinterpret_cast<Acc*>(lds + (mt * 16 + i) * 1024 + (((wave * NT + nt) * 4 + g) ^ i) * 16) = sums;
      }
    __syncthreads();
  }

  // The sums of activation row `row` of the block against its weight rows 4 * piece .. 4 * piece + 3.
  __device__ __forceinline__ Acc sum(int row, int piece) const { return *reinterpret_cast<const Acc*>(lds + row * 1024 + (piece ^ (row & 15)) * 16); }
};

}  // namespace block
}  // namespace dro
