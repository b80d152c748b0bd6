// The matrix-core product of many activation rows (a prompt): a workgroup multiplies a block of activation rows by a
// block of weight rows, both staged through LDS, so that a weight is read and decoded once per block and not once per
// 64 rows.
//
// The sums are tile_mfma.h's to the bit: the same v_mfma instruction on the same k in the same order. In a load step t
// (four 16-byte weight chunks a row) instruction j takes from lane (g, i) the values [8j, 8j + 8) of chunk 4t + g, on both
// sides; a slice of load steps is an ascending f32 chain from zero and the slices' sums are added in ascending order,
// here in a second set of registers (a workgroup walks all of K).
//
// A K tile is 128 bytes of operand a row: 64 values as bf16 (two load steps of bf16 weights, one of the one-byte formats,
// half a step of NVFP4: of every chunk one block of sixteen) or 128 bytes under the byte maths (two steps). In LDS a tile lies
// by pieces of 16 bytes, [piece 4j + g][row]: a fragment read of a 16-lane group is 256 contiguous bytes, the four groups a
// multiple of 256 bytes apart (the LDS's fast pattern), and so are the staging writes, whose 16-lane groups hold sixteen
// rows of one piece. Weights are expanded to bf16 on their way from the staging registers into LDS.
//
// Two LDS buffers, one barrier a tile, two sets of staging registers. Tile t is multiplied from one buffer while tile t + 1 lies
// complete in the other. Its fragments are read ahead, so behind tile t's barrier nobody reads its buffer any more: tile t + 2
// goes there from the registers while tile t + 1's first fragments are read, and tile t + 4 is asked for into those registers.
#pragma once

#include "common.h"
#include "tile_mfma.h"

namespace dro {
namespace block {

// The block <-> workgroup map: consecutive workgroups go to the dies (XCDs) in turn, so workgroup b takes element b / 8 of
// die b % 8's contiguous share of the blocks, and neighbours in that order meet in one die's L2.
__device__ __forceinline__ int die_order(int b, int total) {
  const int die = b & 7, share = total >> 3, extra = total & 7;
  return die * share + min(die, extra) + (b >> 3);
}

// WM x WN wavefronts, each MT x NT tiles of 16 x 16. SPLIT: the row is more than one slice. ONE_X: one set of registers for
// the activations' fragments, each read anew as soon as its products are issued, and the barrier behind a step's first products.
// Reads and products then alternate more evenly and 16 registers are free: the experts' NVFP4 blocks of 128 x 256 at 2048 tokens
// (128 of 4096 x 1536, a pass of the layer) 1476 -> 1388 us; lx_gemm_w's blocks of 128 x 128 are 4 % faster without (fp8 14336 x
// 4096 at 4096 rows 552 / 573, int8 math 4096 x 11008 at 515 rows 162 / 165).
// With SPLIT a 128 x 256 block holds two sets of 64 sums a lane and does not fit 256 registers: the compiler spills 84 .. 200 of
// them (116 .. 180 bytes a lane: the experts in bf16 and NVFP4, lx_gemm_w's on NVFP4 and under the FP8 math), moved where a slice ends. No
// other block spills.
template <int F, int MATH, int WM, int WN, int MT, int NT, bool SPLIT, bool ONE_X = false>
struct Block {
  static constexpr bool kBytes = MATH != LX_MATH_BF16;  // one-byte operands on both sides
  static constexpr int D = 2;  // sets of staging registers (four made no difference: 64 x 64 .. 128 x 128, any row count)
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
  static constexpr int kBufBytes = (BM + BN) * 128;
  static constexpr int kLdsBytes = 2 * kBufBytes;
  static constexpr bool kRaw = F == LX_W_BF16 || kBytes;  // the weights go into LDS as they are: eight 16-byte pieces a tile row
  // Wave-sized units of staging: eight rows by the tile's eight pieces of X; of W the same where it is raw, else sixteen rows by
  // four chunks. (Lanes next to each other hold what is next to each other in memory.) A unit past the last repeats the last.
  static constexpr int kXUnits = BM / 16 * 2, kWUnits = BN / 16 * (kRaw ? 2 : 1);
  static constexpr int XU = (kXUnits + kWaves - 1) / kWaves, WU = (kWUnits + kWaves - 1) / kWaves;
  // bf16 weights: an instruction is a load step, and a slice may end between the two of a tile.
  static constexpr bool kStepHalves = F == LX_W_BF16;
  using Acc = typename std::conditional<MATH == LX_MATH_INT8, i32x4, f32x4>::type;
  using WRaw = typename std::conditional<F == LX_W_NVFP4, u32x2, u32x4>::type;

  struct Set {
    u32x4 x[XU];
    WRaw w[WU];
    uint32_t sc[WU];
  };

  const char* xbase;
  const char* wbase;
  const char* sbase;
  uint32_t xrow[XU], wrow[WU], srow[WU];  // this lane's rows: bytes from the bases
  int xk[XU], wk[WU];                     // its place in a tile's row, in bytes
  uint32_t xput[XU], wput[WU];            // where it goes in a buffer
  int xlast, wlast, slast;                // the last offset a row can be read at
  int K;
  uint8_t* lds;
  int lane, wave;

  // Piece of X (or raw W) at place mp of a tile's row, as an LDS piece 4j + g.
  static __device__ __forceinline__ int piece_of(int mp) {
    if constexpr (F == LX_W_BF16 || kBytes) return mp;
    else return (mp & 1) * 4 + (mp >> 1);
  }

  // How a piece's rows are turned in LDS (row ^ turn). A staging write takes eight lanes at a time, eight pieces of one row
  // (not raw weights: four pieces of two rows), which must fall into eight places mod 8. A fragment read takes half of the
  // lanes of groups g = 0, 1 (2, 3) together, four of every eight rows of one and the others of the other: turns of such a
  // pair may differ in the two low bits only.
  static __device__ __forceinline__ int x_turn(int p) { return p; }
  static __device__ __forceinline__ int w_turn(int p) { return kRaw ? p : 2 * (p & 3); }

  // xoff(row) / woff(row) / soff(row): byte offset of activation row / weight row / weight row's scales (rows of this block,
  // clamped by the caller to rows that exist).
  template <class XOff, class WOff, class SOff>
  __device__ __forceinline__ void init(const void* xb, const void* wb, const void* sb, int64_t row_bytes, int K_, void* lds_, XOff xoff,
                                       WOff woff, SOff soff) {
    lane = threadIdx.x & (kWave - 1);
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    xbase = static_cast<const char*>(xb);
    wbase = static_cast<const char*>(wb);
    sbase = static_cast<const char*>(sb);
    lds = static_cast<uint8_t*>(lds_);
    K = K_;
    xlast = kBytes ? K - 16 : (K - 8) * 2;
    wlast = static_cast<int>(row_bytes) - (F == LX_W_NVFP4 ? 8 : 16);
    slast = K / 16 - 1;
#pragma unroll
    for (int u = 0; u < XU; ++u) {
      const int row = min(u * kWaves + wave, kXUnits - 1) * 8 + (lane >> 3), mp = lane & 7, p = piece_of(mp);
      xrow[u] = xoff(row);
      xk[u] = F == LX_W_NVFP4 ? (mp >> 1) * 64 + (mp & 1) * 16 : mp * 16;
      xput[u] = (p * BM + (row ^ x_turn(p))) * 16;
    }
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      const int v = min(u * kWaves + wave, kWUnits - 1);
      const int row = kRaw ? v * 8 + (lane >> 3) : v * 16 + (lane >> 2), p = kRaw ? lane & 7 : lane & 3;
      wrow[u] = woff(row);
      srow[u] = soff(row);
      wk[u] = p * 16;
      wput[u] = BM * 128 + (p * BN + (row ^ w_turn(p))) * 16;  // not raw: piece (j = 0, g); j = 1 lies 4 * BN * 16 further
    }
  }

  // Bytes from a row's start to K tile kt's first value.
  static __device__ __forceinline__ int xtile(int kt) { return F == LX_W_NVFP4 ? (kt >> 1) * 256 + (kt & 1) * 32 : kt * 128; }
  static __device__ __forceinline__ int wtile(int kt) {
    if constexpr (kRaw) return kt * 128;
    else if constexpr (F == LX_W_NVFP4) return (kt >> 1) * 64 + (kt & 1) * 8;
    else return kt * 64;
  }

  __device__ __forceinline__ void load(Set& s, int kt) const {
    const int xt = xtile(kt), wt = wtile(kt);
#pragma unroll
    for (int u = 0; u < XU; ++u) s.x[u] = *reinterpret_cast<const u32x4*>(xbase + (xrow[u] + static_cast<uint32_t>(min(xt + xk[u], xlast))));
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      s.w[u] = *reinterpret_cast<const WRaw*>(wbase + (wrow[u] + static_cast<uint32_t>(min(wt + wk[u], wlast))));
      if constexpr (F == LX_W_NVFP4)
        s.sc[u] = *reinterpret_cast<const uint8_t*>(sbase + (srow[u] + static_cast<uint32_t>(min((kt >> 1) * 8 + (kt & 1) + (wk[u] >> 3), slast))));
    }
  }

  // Tile kt from the staging registers into a buffer. What lies past K is zero on the activations' side, and in bf16 on the
  // weights' too: a load there repeats the row's last values, and zero times an infinity among them is no zero (the other
  // formats have no infinities). EDGE: the tile may reach past K; bf16 has a loop of its own for the tiles that do not: with one
  // loop the weights' zeros cost 2 % (14336 x 4096 at 4096 rows 593 / 606 us, with two 585). The experts' blocks (ONE_X) have
  // one: 64 experts of 2048 x 1024 at 1024 tokens 398 us, 416 with two.
  template <bool EDGE>
  __device__ __forceinline__ void store_x(const Set& s, int u, int kt, uint8_t* buf) const {
    u32x4 v = s.x[u];
    if (EDGE && xtile(kt) + xk[u] > xlast) v = u32x4{0u, 0u, 0u, 0u};
    *reinterpret_cast<u32x4*>(buf + xput[u]) = v;
  }

  template <bool EDGE>
  __device__ __forceinline__ void store_w(const Set& s, int u, int kt, uint8_t* buf) const {
    if constexpr (kRaw) {
      u32x4 v = s.w[u];
      if (EDGE && F == LX_W_BF16 && wtile(kt) + wk[u] > wlast) v = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(buf + wput[u]) = v;
    } else {
      u32x4 w;
      if constexpr (F == LX_W_NVFP4) w = u32x4{s.w[u].x, s.w[u].y, 0u, 0u};
      else w = s.w[u];
      *reinterpret_cast<bf16x8*>(buf + wput[u]) = weight_fragment<F>(w, s.sc[u], 0);
      *reinterpret_cast<bf16x8*>(buf + wput[u] + 4 * BN * 16) = weight_fragment<F>(w, s.sc[u], 1);
    }
  }

  // Unit u of the staging registers: activations first.
  template <bool EDGE>
  __device__ __forceinline__ void store(const Set& s, int u, int kt, uint8_t* buf) const {
    if (u < XU) store_x<EDGE>(s, u, kt, buf);
    else store_w<EDGE>(s, u - XU, kt, buf);
  }

  // The fragments of a tile's instruction j.
  struct Frags {
    i32x4 x[MT], w[NT];
  };

  __device__ __forceinline__ void fetch_w(Frags& f, const uint8_t* buf, int j) const {
    const uint8_t* const p = buf + BM * 128 + ((4 * j + (lane >> 4)) * BN + wave / WM * NT * 16 + ((lane & 15) ^ w_turn(4 * j + (lane >> 4)))) * 16;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) f.w[nt] = *reinterpret_cast<const i32x4*>(p + nt * 256);
  }

  __device__ __forceinline__ i32x4 fetch_x(const uint8_t* buf, int j, int mt) const {
    const uint8_t* const p = buf + ((4 * j + (lane >> 4)) * BM + wave % WM * 16 + ((lane & 15) ^ x_turn(4 * j + (lane >> 4)))) * 16;
    return *reinterpret_cast<const i32x4*>(p + mt * WM * 256);
  }

  __device__ __forceinline__ void fetch_x(Frags& f, const uint8_t* buf, int j) const {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) f.x[mt] = fetch_x(buf, j, mt);
  }

  static __device__ __forceinline__ void multiply(const i32x4 (&w)[NT], const i32x4& x, int mt, Acc (&acc)[NT][MT]) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if constexpr (kBytes) acc[nt][mt] = byte_mfma<MATH>(w[nt], x, acc[nt][mt]);
      else acc[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[nt]), __builtin_bit_cast(bf16x8, x), acc[nt][mt], 0, 0, 0);
    }
  }

  // The product of `tiles` K tiles from `first` on (a multiple of D; tiles past K count for nothing), in slices of
  // `slice` tiles (kStepHalves: of `slice` load steps, half a tile each). epi(m, tile, sums): the finished sums of the block's activation row m; sums[t][r] belongs to
  // its weight row 16 * (tile + t) + 4 * (lane / 16) + r.
  template <class Epi>
  __device__ __forceinline__ void run(int first, int tiles, int slice, Epi&& epi) {
    Set s[D];
#pragma unroll
    for (int d = 0; d < D; ++d) load(s[d], first + d);
    Acc acc[NT][MT], tot[SPLIT ? NT : 1][SPLIT ? MT : 1];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        acc[nt][mt] = Acc{0, 0, 0, 0};
        if constexpr (SPLIT) tot[nt][mt] = Acc{0, 0, 0, 0};
      }
    uint8_t* const b0 = lds;
    uint8_t* const b1 = lds + kBufBytes;
#pragma unroll
    for (int u = 0; u < XU + WU; ++u) store<true>(s[0], u, first, b0);
    load(s[0], first + D);
#pragma unroll
    for (int u = 0; u < XU + WU; ++u) store<true>(s[1], u, first + 1, b1);
    load(s[1], first + D + 1);
    __syncthreads();
    Frags f0, f1;
    fetch_w(f0, b0, 0);
    fetch_x(f0, b0, 0);
    int flush_at = slice;
    // A slice ends before tile kt (where an instruction is a load step: before instruction `at` of them all).
    auto flush = [&](int at) {
      if constexpr (SPLIT) {
        if (__builtin_expect(at != flush_at, 1)) return;
        flush_at += slice;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            tot[nt][mt] += acc[nt][mt];
            acc[nt][mt] = Acc{0, 0, 0, 0};
          }
      }
    };
    // Tile kt, whose first instruction's fragments are in f0, from `here`. Under their products the second's are read; after
    // the barrier nobody reads `here` any more, and under the second's products tile kt + 1's first fragments are read and
    // tile kt + 2 is written where tile kt was: the writes have half a step until the next barrier waits for them.
    auto step = [&](auto edge, int kt, Set& set, uint8_t* here, const uint8_t* there) {
      flush(kStepHalves ? 2 * kt : kt);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt == 0) fetch_w(f1, here, 1);
        if (mt == (MT > 3 ? 1 : 0)) fetch_x(f1, here, 1);
        multiply(f0.w, f0.x[mt], mt, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
      __syncthreads();
      if constexpr (kStepHalves) flush(2 * kt + 1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt == 0) fetch_w(f0, there, 0);
        if (mt == (MT > 3 ? 1 : 0)) fetch_x(f0, there, 0);
        // The staging units over the groups behind.
        constexpr int kFirst = MT > 1 ? 1 : 0, kGroups = MT - kFirst;
#pragma unroll
        for (int u = 0; u < XU + WU; ++u)
          if (mt == kFirst + u * kGroups / (XU + WU)) store<decltype(edge)::value>(set, u, first + kt + 2, here);
        if (mt == MT - 1) load(set, first + kt + 2 + D);
        multiply(f1.w, f1.x[mt], mt, acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The same with f0.x for both instructions (ONE_X). Tile kt's last fragment is asked for behind the first instruction's last
    // products and used by the second's last; the barrier, which waits for it, stands behind the second's first.
    auto step_one_x = [&](auto edge, int kt, Set& set, uint8_t* here, const uint8_t* there) {
      flush(kStepHalves ? 2 * kt : kt);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if (mt == 0) fetch_w(f1, here, 1);
        multiply(f0.w, f0.x[mt], mt, acc);
        f0.x[mt] = fetch_x(here, 1, mt);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kStepHalves) flush(2 * kt + 1);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        multiply(f1.w, f0.x[mt], mt, acc);
        if (mt == 0) {
          __builtin_amdgcn_sched_barrier(0);
          __syncthreads();
          fetch_w(f0, there, 0);
        }
        f0.x[mt] = fetch_x(there, 0, mt);
#pragma unroll
        for (int u = 0; u < XU + WU; ++u)
          if (mt == u * MT / (XU + WU)) store<decltype(edge)::value>(set, u, first + kt + 2, here);
        if (mt == MT - 1) load(set, first + kt + 2 + D);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto steps = [&](auto edge, int kt) {
#pragma unroll
      for (int d = 0; d < D; ++d)
        if constexpr (ONE_X) step_one_x(edge, kt + d, s[(d + 2) % D], d % 2 ? b1 : b0, d % 2 ? b0 : b1);
        else step(edge, kt + d, s[(d + 2) % D], d % 2 ? b1 : b0, d % 2 ? b0 : b1);
    };
    int kt = 0;
    // Steps kt and kt + 1 write tiles kt + 2 and kt + 3.
    if constexpr (F == LX_W_BF16 && !ONE_X)
      for (const int inside = min(tiles, ((wlast + 16) / 128 - first - 2) & ~1); kt < inside; kt += D) steps(std::false_type{}, kt);
    for (; kt < tiles; kt += D) steps(std::true_type{}, kt);
    const int wm = wave % WM, wn = wave / WM;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      Acc sums[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        sums[nt] = acc[nt][mt];
        if constexpr (SPLIT) sums[nt] = tot[nt][mt] + sums[nt];
      }
      epi((mt * WM + wm) * 16 + (lane & 15), wn * NT, sums);
    }
  }
};

}  // namespace block
}  // namespace dro
