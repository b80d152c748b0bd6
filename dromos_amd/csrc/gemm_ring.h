// lx_gemm_w for a decode step's rows (up to 64) on wide matrices, on block_wide.h's loads: a workgroup takes all of the activation
// rows by BN weight rows, its four wavefronts KS slices of K by 4 / KS parts of the columns. Weights and activations go from memory
// into a ring in LDS that belongs to the wavefront (KS = 4: nothing is shared and nobody waits for anybody) or to the wavefronts of
// a slice. The slices' sums meet in LDS and are added in ascending order; the bits are the other kernels' (tile_mfma.h).
//
// Bound by bytes on their way: a unit's ring holds 80 .. 160 KB of which the activations, which every workgroup reads anew from
// its die's L2, are the larger part from 32 rows on (fp8 14336 x 4096 at 64 rows, 23 us: 17 with the weights alone loaded, 13 with the
// activations alone; the order of a row's lanes, the row stride and the activations asked for ahead make no difference). The
// kernels that stage windows of the activations through registers for all wavefronts (gemm_walk.h) tie or are ahead on many sizes
// (on that one 22.9 / 22.2). Which it takes: gemm.hip, ring_cols().
#pragma once

#include "block_wide.h"
#include "gemm_args.h"

namespace dro {
namespace ring {

using block::Rsrc;
using block::load_to_lds16;
using block::load_to_lds4;
using block::wait_loads;

template <int F, int MT_, int KS_, int BN_>
struct Ring {
  static constexpr int MT = MT_, KS = KS_, BN = BN_;
  static constexpr bool kNv = F == LX_W_NVFP4, kRaw = F == LX_W_BF16;
  static constexpr int kWaves = 4, kThreads = kWaves * kWave, WN = kWaves / KS, NT = BN / 16 / WN;
  static_assert(NT >= 1, "a tile of weight rows a wavefront at least");
  static constexpr int BM = MT * 16;
  static constexpr int kSteps = kRaw ? 2 : 1;  // load steps a stage
  static constexpr int J = kNv ? 4 : 2;
  static constexpr int kXRow = kNv ? 256 : 128, kWRow = kRaw ? 128 : 64;
  // Wave-sized loads a stage and wavefront: its part of its slice's activations, its own weights and block scales.
  static constexpr int kXLoads = (BM * kXRow / 1024 + WN - 1) / WN, kWLoads = NT * 16 * kWRow / 1024, kSLoads = kNv ? (NT + 1) / 2 : 0;
  static constexpr int kLoads = kXLoads + kWLoads + kSLoads;
  static constexpr int kXBytes = kXLoads * WN * 1024, kWBytes = kWLoads * 1024, kOwn = kWBytes + kSLoads * 256;
  static constexpr int kStage = KS * kXBytes + kWaves * kOwn;
  // Where in a stage: a slice's activations, which its WN wavefronts load and read; what one wavefront alone loads and reads; and
  // (NVFP4, in the ring's last stage) where a wavefront's look-ahead goes, 256 bytes.
  static constexpr int x_at(int ks) { return ks * kXBytes; }
  static constexpr int own_at(int wave) { return KS * kXBytes + wave * kOwn; }
  static constexpr int ahead_at(int wave) { return own_at(wave); }
  static_assert(kOwn >= 256, "room for a look-ahead");
  static constexpr int fit(int a, int b) { return a < b ? a : b; }
  static constexpr int kStages = fit(fit(160 * 1024 / kStage, 8), 63 / kLoads + 2);
  static constexpr bool kFits = kStages >= 2;
  static constexpr int kSums = KS * BM * BN * 4;
  static constexpr int kLdsBytes = kStages * kStage > kSums ? kStages * kStage : kSums;
};

// What a kernel below leaves in LDS, SL slices' sums of BM rows by BN columns side by side, added up in ascending order and written out by
// THREADS threads.
template <int F, int BM, int BN, int SL, int THREADS>
__device__ __forceinline__ void write_slices(const GemmArgs& a, const uint8_t* lds, int n0, int cols, int slices) {
  constexpr int kPieces = BN / 4, kSlice = BM * BN * 4;
  const int piece = threadIdx.x % kPieces, n = 4 * piece;
  if (n >= cols) return;
  const bool wide = wide_stores(a) && n + 3 < cols;
  constexpr int kRows = THREADS / kPieces, kTimes = (BM + kRows - 1) / kRows;
  float rf[4], xs[kTimes];
#pragma unroll
  for (int r = 0; r < 4; ++r) rf[r] = row_factor(F, a.scale, a.global, n0 + min(n + r, cols - 1));
#pragma unroll
  for (int q = 0; q < kTimes; ++q) xs[q] = a.act_scale ? a.act_scale[min(static_cast<int>(threadIdx.x) / kPieces + q * kRows, a.M - 1)] : 1.0f;
#pragma unroll
  for (int q = 0; q < kTimes; ++q) {
    const int m = threadIdx.x / kPieces + q * kRows;
    if (m >= a.M || m >= BM) break;
    const uint8_t* const at = lds + m * BN * 4 + ((piece ^ (m & 15)) & (kPieces - 1)) * 16;
    f32x4 s = *reinterpret_cast<const f32x4*>(at);
#pragma unroll
    for (int k = 1; k < SL; ++k)
      if (k < slices) s += *reinterpret_cast<const f32x4*>(at + k * kSlice);
    float f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = rf[r] * xs[q];
    if (wide) write_four(a, m * a.ld_y + n0 + n, s, f);
    else write_each(a, m, n0 + n, s, f);
  }
}

template <int F, int MT, int KS, int BN>
__global__ void __launch_bounds__(4 * kWave) __attribute__((amdgpu_waves_per_eu(1, 2))) ring_kernel(const GemmArgs a, int slices) {
  using R = Ring<F, MT, KS, BN>;
  constexpr int WN = R::WN, NT = R::NT, J = R::J, kStages = R::kStages, kLoads = R::kLoads;
  extern __shared__ __align__(16) f32x4 lds4[];
  uint8_t* const lds = reinterpret_cast<uint8_t*>(lds4);
  const uint32_t lds_at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds)));
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), g = lane >> 4, i = lane & 15;
  const int ks = wave % KS, wn = wave / KS;
  const int n0 = blockIdx.x * BN, cols = min(BN, a.N - n0);
  const int xbytes = a.K * 2, wbytes = static_cast<int>(a.row_bytes), sbytes = a.K / 16;
  const int64_t ld = a.xs.ld * 2;
  const Rsrc xbuf = block::buffer_of(a.xs.x, (a.M - 1) * ld + xbytes), wbuf = block::buffer_of(a.w + n0 * a.row_bytes, cols * a.row_bytes),
             sbuf = block::buffer_of(R::kNv ? a.scale + n0 * a.scale_row_bytes : a.scale, cols * a.scale_row_bytes);
  // This slice's stages (all slices walk as many; what lies past the row's end is zero), and the last one with anything in it.
  const int per = a.steps_per_wave / R::kSteps, first = ks * per, end = (a.steps + R::kSteps - 1) / R::kSteps - 1;
  uint32_t xrow[R::kXLoads], wrow[R::kWLoads], srow[R::kSLoads > 0 ? R::kSLoads : 1];
  int xpiece = 0, wpiece = 0;
  const int spiece = (lane & 1) * 4;
  // Places in a row as in block_wide.h: slot s of activation row r holds place s ^ r (instruction p / 4's, lane group p % 4's); of a
  // weight row piece s ^ (r / 2), of a bf16 weight row s ^ r.
#pragma unroll
  for (int u = 0; u < R::kXLoads; ++u) {
    constexpr int kSlots = R::kXRow / 16;
    const int at = (u * WN + wn) * kWave + lane, row = at / kSlots, place = (at ^ row) % kSlots;
    xpiece = (R::kRaw ? place : J * (place & 3) + (place >> 2)) * 16;
    xrow[u] = static_cast<uint32_t>(min(row, a.M - 1)) * static_cast<uint32_t>(ld) + xpiece;
  }
#pragma unroll
  for (int u = 0; u < R::kWLoads; ++u) {
    constexpr int kSlots = R::kWRow / 16;
    const int at = u * kWave + lane, row = at / kSlots;
    wpiece = ((at % kSlots) ^ (R::kRaw ? row & 7 : (row >> 1) & 3)) * 16;
    wrow[u] = static_cast<uint32_t>(min(wn * NT * 16 + row, cols - 1)) * static_cast<uint32_t>(wbytes) + wpiece;
  }
#pragma unroll
  for (int u = 0; u < R::kSLoads; ++u)
    srow[u] = static_cast<uint32_t>(min(wn * NT * 16 + min(u * 32 + (lane >> 1), NT * 16 - 1), cols - 1)) * static_cast<uint32_t>(a.scale_row_bytes) + spiece;
  const uint32_t x_at = R::x_at(ks), own_at = R::own_at(wave);  // in a stage
  // Load u of the slice's stage st: what lies past the row's end is asked for at its start (its last stage's) and zeroed by finish().
  auto load = [&](int st, int slot, int u) {
    const int t = min(first + st, end);
    const uint32_t to = lds_at + slot * R::kStage;
    if (u < R::kWLoads) {
      load_to_lds16(to + own_at + u * 1024, wrow[u] - (wpiece + t * R::kWRow >= wbytes ? wpiece : 0), wbuf, t * R::kWRow);
    } else if (u < R::kWLoads + R::kSLoads) {
      load_to_lds4(to + own_at + R::kWBytes + (u - R::kWLoads) * 256, srow[u - R::kWLoads] - (spiece + t * 8 >= sbytes ? spiece : 0), sbuf, t * 8);
    } else {
      const int v = u - R::kWLoads - R::kSLoads;
      load_to_lds16(to + x_at + (v * WN + wn) * 1024, xrow[v] - (xpiece + t * R::kXRow >= xbytes ? xpiece : 0), xbuf, t * R::kXRow);
    }
  };
  auto finish = [&](int st, int slot) {
    uint8_t* const to = lds + slot * R::kStage;
    const int t = first + st;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    if (xpiece + static_cast<int64_t>(t) * R::kXRow >= xbytes) {
#pragma unroll
      for (int u = 0; u < R::kXLoads; ++u) *reinterpret_cast<u32x4*>(to + x_at + (u * WN + wn) * 1024 + lane * 16) = zero;
    }
    if (wpiece + static_cast<int64_t>(t) * R::kWRow >= wbytes) {
#pragma unroll
      for (int u = 0; u < R::kWLoads; ++u) *reinterpret_cast<u32x4*>(to + own_at + u * 1024 + lane * 16) = zero;
    }
#pragma unroll
    for (int u = 0; u < R::kSLoads; ++u) {
      if (spiece + t * 8 >= sbytes) *reinterpret_cast<uint32_t*>(to + own_at + R::kWBytes + u * 256 + lane * 4) = 0;  // (four bytes are all or none of a row)
    }
  };
  uint32_t xat[J];
#pragma unroll
  for (int j = 0; j < J; ++j) xat[j] = x_at + i * R::kXRow + ((4 * j + g) ^ (i % (R::kXRow / 16))) * 16;
  const uint32_t wat = own_at + i * R::kWRow + (R::kRaw ? g ^ (i & 7) : g ^ ((i >> 1) & 3)) * 16, sat = own_at + R::kWBytes + i * 8 + g * 2;
  f32x4 acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 raw[NT], wf[2][NT], xf[2][MT];
  uint32_t sc[NT];
  auto fetch_raw = [&](const uint8_t* st, int nt) {
    sc[nt] = 0;
    if constexpr (!R::kRaw) raw[nt] = *reinterpret_cast<const u32x4*>(st + wat + nt * 16 * R::kWRow);
    if constexpr (R::kNv) sc[nt] = *reinterpret_cast<const uint16_t*>(st + sat + nt * 128);
  };
  auto fetch_w = [&](u32x4(&w)[NT], const uint8_t* st, int j, int nt) {
    if constexpr (R::kRaw) w[nt] = *reinterpret_cast<const u32x4*>(st + (wat ^ (j ? 64 : 0)) + nt * 16 * R::kWRow);
    else
#pragma unroll
      for (int p = 0; p < 4; ++p) w[nt][p] = block::weight_pair<F>(raw[nt], sc[nt], j, p);
  };
  auto fetch_x = [&](u32x4(&x)[MT], const uint8_t* st, int j, int mt) { x[mt] = *reinterpret_cast<const u32x4*>(st + xat[j] + mt * 16 * R::kXRow); };
  // Stage st is here: this wavefront's loads, and the others' of the slice.
  auto arrive = [&](auto steady, int st, int slot) {
    if constexpr (decltype(steady)::value) {
      wait_loads<(kStages - 2) * kLoads>();
    } else {
      const int behind = min(per - 1 - st, kStages - 2);
      if (behind == kStages - 2) wait_loads<(kStages - 2) * kLoads>();
      else if (behind == 1) wait_loads<kLoads>();
      else if (kStages > 4 && behind == 2) wait_loads<(kStages > 4 ? 2 : 0) * kLoads>();
      else if (kStages > 5 && behind == 3) wait_loads<(kStages > 5 ? 3 : 0) * kLoads>();
      else if (kStages > 6 && behind == 4) wait_loads<(kStages > 6 ? 4 : 0) * kLoads>();
      else if (kStages > 7 && behind == 5) wait_loads<(kStages > 7 ? 5 : 0) * kLoads>();
      else wait_loads<0>();
    }
    if (first + st >= end) {  // (the row may end inside it, or before it)
      finish(st, slot);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    if constexpr (WN > 1) asm volatile("s_barrier" ::: "memory");
  };
  // All workgroups walk K together, so an activation row's next piece would come from memory for every one of them. The workgroups
  // of a die (every eighth) share out the activations' 128-byte lines and ask for them once, at the start: the walk then finds
  // them in the die's L2. They land in the wavefront's own part of the ring's last slot: with a slice a wavefront nobody waits for
  // anybody else's loads, and its own stage kStages - 1 is asked for behind a wait for these. NVFP4 8192 x 8192 at
  // 33 rows 23.7 -> 22.8 us; one-byte weights lose 4 .. 6 %.
  if constexpr (R::kNv) {
    const int line_row = (xbytes + 127) / 128, lines = line_row * a.M, share = (lines + (gridDim.x >> 3)) / ((gridDim.x >> 3) + 1);
    for (int at = static_cast<int>(threadIdx.x); at - lane < share; at += R::kThreads) {
      const int line = min(static_cast<int>(blockIdx.x >> 3) * share + min(at, share - 1), lines - 1), row = line / line_row;
      load_to_lds4(lds_at + (kStages - 1) * R::kStage + R::ahead_at(wave), static_cast<uint32_t>(row) * static_cast<uint32_t>(ld) + (line - row * line_row) * 128, xbuf, 0);
    }
  }
#pragma unroll
  for (int st = 0; st < kStages - 1; ++st)
    if (st < per) {
#pragma unroll
      for (int u = 0; u < kLoads; ++u) load(st, st, u);
    }
  arrive(std::false_type{}, 0, 0);
  if (kStages - 1 < per) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) load(kStages - 1, kStages - 1, u);
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    fetch_raw(lds, nt);
    fetch_w(wf[0], lds, 0, nt);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) fetch_x(xf[0], lds, 0, mt);
  int slot = 0;
  // As block_wide.h's step: under an instruction's products the next one's fragments are read and expanded.
  auto step = [&](auto steady, int st) {
    const int next = slot + 1 == kStages ? 0 : slot + 1;
    const uint8_t *const here = lds + slot * R::kStage, *const there = lds + next * R::kStage;
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const bool last = j == J - 1;
      const uint8_t* const from = last ? there : here;
      __builtin_amdgcn_sched_barrier(0);
      if (last) {
        if (decltype(steady)::value || st + 1 < per) arrive(steady, st + 1, next);
        if constexpr (decltype(steady)::value) {
#pragma unroll
          for (int u = 0; u < kLoads; ++u) load(st + kStages, slot, u);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) fetch_raw(from, nt);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) fetch_x(xf[(j + 1) & 1], from, (j + 1) % J, mt);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[j & 1][nt]), __builtin_bit_cast(bf16x8, xf[j & 1][mt]), acc[nt][mt], 0, 0, 0);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) fetch_w(wf[(j + 1) & 1], from, (j + 1) % J, nt);
#pragma unroll
      for (int n = 0; n < MT * NT; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, R::kNv ? 4 : 3, 0);
      }
    }
    slot = next;
  };
  int st = 0;
  for (; st + kStages < per; ++st) step(std::true_type{}, st);
  for (; st < per; ++st) step(std::false_type{}, st);
  __builtin_amdgcn_sched_barrier(0);
  // The slices' sums side by side in LDS, a row's pieces of four turned by the row; then everyone adds up what it writes.
  constexpr int kPieces = BN / 4, kSlice = R::BM * BN * 4;
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      *reinterpret_cast<f32x4*>(lds + ks * kSlice + (mt * 16 + i) * BN * 4 + ((((wn * NT + nt) * 4 + g) ^ i) & (kPieces - 1)) * 16) = acc[nt][mt];
  __syncthreads();
  write_slices<F, R::BM, BN, KS, R::kThreads>(a, lds, n0, cols, slices);
}

// The same product on NVFP4 weights with the loads on wavefronts of their own: of a workgroup's eight, four multiply (two slices by two
// parts of 64 columns; PER slices one after the other), two load a slice's activations each and two its weights (the feeders). A wavefront's
// loads return in the order they were asked for, so in ring_kernel the activations, which come from the die's L2, wait behind weights from
// memory; here the two wait apart, and the weights' ring is as deep as LDS allows. What the row does not fill of the last slices is not
// walked (ring_kernel multiplies zeros there).
// 14336 x 4096 at 64 rows 28.3 -> 21.1 us (by gemm_walk.h before), 16384 x 4096 28.4 -> 21.0, 8256 x 4416 at 50 rows 67 -> 26 (by the windows before).
// Bound by no one thing. Counters of that launch (45500 cycles): a SIMD issues in half of them at most (its multiplying wavefront about 220 vector
// instructions a stage, 32 of them matrix instructions and 128 conversions, and 22 LDS reads; its feeder hardly any), the matrix cores are busy in 0.18,
// LDS in 0.13, without a bank conflict. A third is the launch, the first loads and the sums' way out, and the walk waits for memory besides: with
// every load from one row, out of L2, 16.7 us. (The loads on the multiplying wavefronts the same time at 64 rows and 1 us more at 32; a stage's
// codes read a quarter earlier 1 us more.)
// A barrier a stage: behind stage st's it is in LDS, and nobody reads stage st - 1 any more.
template <int MT_, int PER_>
struct Fed {
  static constexpr int MT = MT_, PER = PER_, KS = 2, BN = 64;
  using R = Ring<LX_W_NVFP4, MT, KS, BN>;
  static_assert(R::WN == 2 && R::NT == 2);
  static constexpr int kThreads = 2 * R::kThreads;
  // A stage: the slices' activations; of weights the multiplying wavefronts' parts, codes and block scales.
  static constexpr int kXStage = KS * R::kXBytes, kWStage = R::kWaves * R::kOwn;
  static constexpr int kXL = R::kXLoads * R::WN, kWL = (R::kWLoads + R::kSLoads) * R::WN;  // a feeder's loads a stage
  static constexpr int fit(int a, int b) { return a < b ? a : b; }
  static constexpr int kXStages = MT == 4 ? 3 : 4;
  static constexpr int kWAt = kXStages * kXStage;
  static constexpr int kWStages = fit(fit((160 * 1024 - kWAt) / kWStage, 10), 63 / kWL + 1);
  static_assert(kXStages <= 63 / kXL + 2 && kWStages >= 3);
  static constexpr int kSums = KS * PER * R::BM * BN * 4, kRing = kWAt + kWStages * kWStage, kLdsBytes = kRing > kSums ? kRing : kSums;
};

// What a feeder's walk does on the device: load(st, slot) asks for stage st's loads, finish(st, slot) writes zeros where a stage reaches past
// the row's end. (A walk of its own because tests follow it on the host: gemm.hip, dromos_feed_in_flight().)
template <class Load, class Finish>
struct Feeder {
  Load load;
  Finish finish;
  template <int LEFT>
  __device__ __forceinline__ void wait() const {
    wait_loads<LEFT>();
  }
  __device__ __forceinline__ void written() const { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
  __device__ __forceinline__ void barrier() const { asm volatile("s_barrier" ::: "memory"); }
};
template <class Load, class Finish>
__device__ __forceinline__ Feeder<Load, Finish> feeder(Load load, Finish finish) {
  return {load, finish};
}

// Waits until at most `behind` (0 .. MOST) stages of L loads each are on their way.
template <int L, int MOST, class Walk>
__host__ __device__ __forceinline__ void wait_stages(int behind, Walk& walk) {
  if constexpr (MOST == 0) walk.template wait<0>();
  else if (behind >= MOST) walk.template wait<MOST * L>();
  else wait_stages<L, MOST - 1>(behind, walk);
}

// A feeder's walk over `stages` stages of L loads each by a ring of STAGES; stage `cut` is finished once it has arrived. `all` stages have a
// barrier. Whatever was asked for before the walk (a look-ahead) is here when it ends, as the walk's own loads are: a feeder that has no
// stage has waited for nothing else, and behind the walk the ring's bytes are the sums'.
template <int L, int STAGES, class Walk>
__host__ __device__ __forceinline__ void feed(int stages, int all, int cut, Walk&& walk) {
  for (int st = 0; st < STAGES - 1; ++st)
    if (st < stages) walk.load(st, st);
  int slot = 0, free = STAGES - 1;  // stage st's slot, and the one that stage st - 1 + STAGES takes
  for (int st = 0; st < stages; ++st) {
    wait_stages<L, STAGES - 2>(stages - 1 - st, walk);
    if (st == cut) {
      walk.finish(st, slot);
      walk.written();
    }
    walk.barrier();
    if (st - 1 + STAGES < stages) walk.load(st - 1 + STAGES, free);
    slot = slot + 1 == STAGES ? 0 : slot + 1;
    free = free + 1 == STAGES ? 0 : free + 1;
  }
  for (int st = stages; st < all; ++st) walk.barrier();
  walk.template wait<0>();
}

template <int MT, int PER>
__global__ void __launch_bounds__(8 * kWave) __attribute__((amdgpu_waves_per_eu(2, 2))) fed_kernel(const GemmArgs a, int slices) {
  using D = Fed<MT, PER>;
  using R = typename D::R;
  constexpr int F = LX_W_NVFP4, WN = R::WN, NT = R::NT, J = R::J, KS = D::KS, BN = D::BN;
  extern __shared__ __align__(16) f32x4 lds4[];
  uint8_t* const lds = reinterpret_cast<uint8_t*>(lds4);
  const uint32_t lds_at = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t*)lds)));
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), g = lane >> 4, i = lane & 15;
  const int ks = wave % KS, wn = wave / KS % WN;
  const int n0 = blockIdx.x * BN, cols = min(BN, a.N - n0);
  const int xbytes = a.K * 2, wbytes = static_cast<int>(a.row_bytes), sbytes = a.K / 16;
  const int64_t ld = a.xs.ld * 2;
  // The stages of this wavefront's slices, and those of them that the row has (the others are barriers only). The row's last one, `end`,
  // may be cut short by K: zeros there.
  const int per = PER * a.steps_per_wave, first = ks * per, end = a.steps - 1, stages = max(0, min(per, a.steps - first));
  constexpr int kSlice = R::BM * BN * 4;
  if (wave >= R::kWaves + KS) {
    // Slice ks's weights and block scales, for the WN wavefronts that multiply them; a stage is a load step, 64 bytes of a row (8 of scales).
    const Rsrc wbuf = block::buffer_of(a.w + n0 * a.row_bytes, cols * a.row_bytes), sbuf = block::buffer_of(a.scale + n0 * a.scale_row_bytes, cols * a.scale_row_bytes);
    const int wpiece = ((lane & 3) ^ ((lane >> 3) & 3)) * 16, spiece = (lane & 1) * 4;  // piece s ^ (r / 2) of row r at slot s, as in ring_kernel
    uint32_t wrow[WN][R::kWLoads], srow[WN];
    static_assert(R::kWRow == 64 && R::kSLoads == 1 && NT * 16 == 32);
#pragma unroll
    for (int h = 0; h < WN; ++h) {
#pragma unroll
      for (int u = 0; u < R::kWLoads; ++u)
        wrow[h][u] = static_cast<uint32_t>(min(h * 32 + u * 16 + (lane >> 2), cols - 1)) * static_cast<uint32_t>(wbytes) + wpiece;
      srow[h] = static_cast<uint32_t>(min(h * 32 + (lane >> 1), cols - 1)) * static_cast<uint32_t>(a.scale_row_bytes) + spiece;
    }
    feed<D::kWL, D::kWStages>(
        stages, per, end - first,
        feeder([&](int st, int slot) {
          const int t = first + st;
          const uint32_t to = lds_at + D::kWAt + slot * D::kWStage + ks * R::kOwn;
          const uint32_t wback = wpiece + t * 64 >= wbytes ? wpiece : 0, sback = spiece + t * 8 >= sbytes ? spiece : 0;
#pragma unroll
          for (int h = 0; h < WN; ++h) {
#pragma unroll
            for (int u = 0; u < R::kWLoads; ++u) load_to_lds16(to + h * KS * R::kOwn + u * 1024, wrow[h][u] - wback, wbuf, t * 64);
            load_to_lds4(to + h * KS * R::kOwn + R::kWBytes, srow[h] - sback, sbuf, t * 8);
          }
        },
        [&](int st, int slot) {
          const int t = first + st;
#pragma unroll
          for (int h = 0; h < WN; ++h) {
            uint8_t* const to = lds + D::kWAt + slot * D::kWStage + (h * KS + ks) * R::kOwn;
            if (wpiece + t * 64 >= wbytes) {
#pragma unroll
              for (int u = 0; u < R::kWLoads; ++u) *reinterpret_cast<u32x4*>(to + u * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
            }
            if (spiece + t * 8 >= sbytes) *reinterpret_cast<uint32_t*>(to + R::kWBytes + lane * 4) = 0;  // (four bytes are all or none of a row)
          }
        }));
  } else if (wave >= R::kWaves) {
    // Slice ks's activations, 256 bytes of every row a stage. Places in a row as in ring_kernel.
    const Rsrc xbuf = block::buffer_of(a.xs.x, (a.M - 1) * ld + xbytes);
    uint32_t xrow[D::kXL];
    int xpiece[4];
    static_assert(R::kXRow == 256 && J == 4 && D::kXL >= 4);
#pragma unroll
    for (int u = 0; u < D::kXL; ++u) {
      const int row = u * 4 + (lane >> 4), place = (lane ^ row) & 15;
      const int piece = (J * (place & 3) + (place >> 2)) * 16;
      if (u < 4) xpiece[u] = piece;  // (the same for every sixteen rows)
      xrow[u] = static_cast<uint32_t>(min(row, a.M - 1)) * static_cast<uint32_t>(ld) + piece;
    }
    const uint32_t own = ks * R::kXBytes;
    // All workgroups walk K together, so an activation row's next piece would come from memory for every one of them. The workgroups of
    // a die (every eighth) share out the activations' 128-byte lines and ask for them once, at the start. They land where this
    // feeder loads the last slot's stage, which it asks for behind a wait for these (a feeder without stages waits at its walk's end).
    {
      const int line_row = (xbytes + 127) / 128, lines = line_row * a.M, share = (lines + (gridDim.x >> 3)) / ((gridDim.x >> 3) + 1);
      for (int at = ks * kWave + lane; at - lane < share; at += KS * kWave) {
        const int line = min(static_cast<int>(blockIdx.x >> 3) * share + min(at, share - 1), lines - 1), row = line / line_row;
        load_to_lds4(lds_at + (D::kXStages - 1) * D::kXStage + own, static_cast<uint32_t>(row) * static_cast<uint32_t>(ld) + (line - row * line_row) * 128, xbuf, 0);
      }
    }
    feed<D::kXL, D::kXStages>(
        stages, per, end - first,
        feeder([&](int st, int slot) {
          const int t = first + st;
          uint32_t back[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) back[q] = xpiece[q] + t * 256 >= xbytes ? xpiece[q] : 0;
#pragma unroll
          for (int u = 0; u < D::kXL; ++u) load_to_lds16(lds_at + slot * D::kXStage + own + u * 1024, xrow[u] - back[u & 3], xbuf, t * 256);
        },
        [&](int st, int slot) {
#pragma unroll
          for (int u = 0; u < D::kXL; ++u)
            if (xpiece[u & 3] + (first + st) * 256 >= xbytes)
              *reinterpret_cast<u32x4*>(lds + slot * D::kXStage + own + u * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
        }));
  }
  if (wave >= R::kWaves) {
    __syncthreads();
  } else {
    uint32_t xat[J];
#pragma unroll
    for (int j = 0; j < J; ++j) xat[j] = ks * R::kXBytes + i * R::kXRow + ((4 * j + g) ^ i) * 16;
    const uint32_t own = D::kWAt + wave * R::kOwn, wat = own + i * 64 + (g ^ ((i >> 1) & 3)) * 16, sat = own + R::kWBytes + i * 8 + g * 2;
    f32x4 acc[NT][MT], done[PER][NT][MT];  // the slice at hand, and the slices walked
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 raw[NT], wf[2][NT], xf[2][MT];
    uint32_t sc[NT];
    auto fetch_raw = [&](const uint8_t* st, int nt) {
      raw[nt] = *reinterpret_cast<const u32x4*>(st + wat + nt * 1024);
      sc[nt] = *reinterpret_cast<const uint16_t*>(st + sat + nt * 128);
    };
    auto fetch_w = [&](u32x4(&w)[NT], int j, int nt) {
#pragma unroll
      for (int p = 0; p < 4; ++p) w[nt][p] = block::weight_pair<F>(raw[nt], sc[nt], j, p);
    };
    auto fetch_x = [&](u32x4(&x)[MT], const uint8_t* st, int j, int mt) { x[mt] = *reinterpret_cast<const u32x4*>(st + xat[j] + mt * 16 * R::kXRow); };
    // (What was read of the stage before is in registers.)
    auto arrive = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    arrive();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      fetch_raw(lds, nt);
      fetch_w(wf[0], 0, nt);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) fetch_x(xf[0], lds, 0, mt);
    const uint8_t *x_here = lds, *w_here = lds;  // the stage's slots
    const uint8_t *const x_end = lds + D::kXStages * D::kXStage, *const w_end = lds + D::kWStages * D::kWStage;
    int st = 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      for (const int all = min((q + 1) * a.steps_per_wave, stages); st < all; ++st) {
        const uint8_t *x_next = x_here + D::kXStage, *w_next = w_here + D::kWStage;
        x_next = x_next == x_end ? lds : x_next;
        w_next = w_next == w_end ? lds : w_next;
        // As block_wide.h's step: under an instruction's products the next one's fragments are read and expanded.
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const bool last = j == J - 1;
          __builtin_amdgcn_sched_barrier(0);
          if (last) {
            if (st + 1 < stages) arrive();
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) fetch_raw(w_next, nt);
          }
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) fetch_x(xf[(j + 1) & 1], last ? x_next : x_here, (j + 1) % J, mt);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
              acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[j & 1][nt]), __builtin_bit_cast(bf16x8, xf[j & 1][mt]), acc[nt][mt], 0, 0, 0);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) fetch_w(wf[(j + 1) & 1], (j + 1) % J, nt);
#pragma unroll
          for (int n = 0; n < MT * NT; ++n) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
          }
        }
        x_here = x_next;
        w_here = w_next;
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          done[q][nt][mt] = acc[nt][mt];
          acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    for (int b = max(stages, 1); b < per; ++b) asm volatile("s_barrier" ::: "memory");
    __syncthreads();
    // The slices' sums side by side in LDS, a row's pieces of four turned by the row; then everyone adds up what it writes.
#pragma unroll
    for (int q = 0; q < PER; ++q)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          *reinterpret_cast<f32x4*>(lds + (ks * PER + q) * kSlice + (mt * 16 + i) * BN * 4 + ((((wn * NT + nt) * 4 + g) ^ i) & (BN / 4 - 1)) * 16) = done[q][nt][mt];
  }
  __syncthreads();
  write_slices<F, R::BM, BN, KS * PER, D::kThreads>(a, lds, n0, cols, slices);
}

template <class R, int F>
int launch(const GemmArgs& a, int slices, hipStream_t stream) {
  const auto kernel = ring_kernel<F, R::MT, R::KS, R::BN>;
  allow_lds(reinterpret_cast<const void*>(kernel), R::kLdsBytes);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((a.N + R::BN - 1) / R::BN)), dim3(R::kThreads), R::kLdsBytes, stream, a, slices);
  return status_of(hipGetLastError());
}

// fn(the Ring for M rows in `slices` slices with `cols` (32 or 64) weight rows a workgroup); false where ring_cols() has no such call: only
// NVFP4 rows are ever cut in two, only bf16 weights taken at 16 rows and fewer, one-byte weights with 64 columns from 33 rows.
template <int F, class Fn>
bool with_ring(int M, int slices, int cols, Fn&& fn) {
  auto rows = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    if (slices < 2 || slices > 4) return false;
    if (slices == 2) {
      if constexpr (F == LX_W_NVFP4) {
        if (cols == 32) fn(Ring<F, MT, 2, 32>{});
        else fn(Ring<F, MT, 2, 64>{});
        return true;
      }
      return false;
    }
    if (cols == 32) {
      fn(Ring<F, MT, 4, 32>{});
      return true;
    }
    if constexpr (Ring<F, MT, 4, 64>::kFits && (MT > 2 || F == LX_W_BF16 || F == LX_W_NVFP4)) {
      fn(Ring<F, MT, 4, 64>{});
      return true;
    }
    return false;
  };
  switch ((M + 15) / 16) {
    case 1:
      if constexpr (F == LX_W_BF16) return rows(std::integral_constant<int, 1>{});
      return false;
    case 2: return rows(std::integral_constant<int, 2>{});
    case 3: return rows(std::integral_constant<int, 3>{});
    default: return rows(std::integral_constant<int, 4>{});
  }
}

template <int F>
bool launch_ring(const GemmArgs& a, int cols, int* status, hipStream_t stream) {
  const int slices = (a.steps + a.steps_per_wave - 1) / a.steps_per_wave;
  return with_ring<F>(a.M, slices, cols, [&](auto ring) { *status = launch<decltype(ring), F>(a, slices, stream); });
}

template <int MT, int PER>
int launch_fed_as(const GemmArgs& a, int slices, hipStream_t stream) {
  using D = Fed<MT, PER>;
  const auto kernel = fed_kernel<MT, PER>;
  allow_lds(reinterpret_cast<const void*>(kernel), D::kLdsBytes);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((a.N + D::BN - 1) / D::BN)), dim3(D::kThreads), D::kLdsBytes, stream, a, slices);
  return status_of(hipGetLastError());
}

inline int launch_fed(const GemmArgs& a, hipStream_t stream) {
  const int slices = (a.steps + a.steps_per_wave - 1) / a.steps_per_wave;
  auto go = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    return slices > 2 ? launch_fed_as<MT, 2>(a, slices, stream) : launch_fed_as<MT, 1>(a, slices, stream);
  };
  switch ((a.M + 15) / 16) {
    case 1:
    case 2: return go(std::integral_constant<int, 2>{});
    case 3: return go(std::integral_constant<int, 3>{});
    default: return go(std::integral_constant<int, 4>{});
  }
}

}  // namespace ring
}  // namespace dro
