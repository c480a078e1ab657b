// Shared pieces of the FP8, NVFP4 and BF16 (over Q4_K) GEMMs: staging by direct
// global->LDS copies, the waits of the rings, the bank conflict check, the tile
// cost rule and the stores. Tile and ring() are those of FP8 and NVFP4, which
// multiply two operands of the same 128-byte-per-row K chunks (128 E4M3
// codes, or 256 E2M1 nibbles) on FP16 MFMAs and widen the raw bytes to FP16 in
// registers, fragment by fragment; prefill_bf16.hip has its own.
//
// LDS image of an FP8 or NVFP4 operand: row R at 128 R, its eight 16-byte pieces permuted
// by an XOR key so that the b128 fragment reads are free of bank conflicts
// (b128_clean). MFMA lane (lr, lk)
// takes piece 4 h + lk (h = 0, 1) whole, for both operands: which K index an
// MFMA slot holds is then a permutation of the chunk common to both sides.
#pragma once

#include <iterator>
#include <type_traits>

#include "lowp.hpp"

namespace qw38hip {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));

// Wait until at most N of this wave's copies are in flight and its LDS reads
// have returned, then the workgroup barrier.
template <int N>
__device__ __forceinline__ void copies_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Whether a wave's b128 LDS access (addr: byte address of a lane) is free of
// bank conflicts: the 64 banks serve it in groups of 16 lanes, {0-3, 12-15, 20-27}, the
// other half of the first 32 lanes, and the same of the last 32, and a group's
// different addresses must lie in different 16-byte slots of 256. (Measured with
// eight waves of a CU: 1.8 ns per read, 3.4 ns with pairs in one slot.)
template <class F>
__host__ __device__ constexpr bool b128_clean(F addr) {
  for (uint32_t g = 0; g < 4; ++g)
    for (uint32_t i = 0; i < 32; ++i)
      for (uint32_t j = 0; j < i; ++j) {
        auto second = [](uint32_t l) { return (l >= 4 && l < 12) || (l >= 16 && l < 20) || l >= 28; };
        if (second(i) != bool(g & 1u) || second(j) != bool(g & 1u)) continue;
        const uint32_t a = addr(g / 2 * 32 + i), b = addr(g / 2 * 32 + j);
        if (a != b && a / 16 % 16 == b / 16 % 16) return false;
      }
  return true;
}

// 16 bytes from an address of any alignment, in one load instruction (gfx950
// takes unaligned global addresses).
__device__ __forceinline__ u4 load16(const uint8_t* g) {
  u4 v;
  __builtin_memcpy(&v, g, 16);
  return v;
}

// A lane's 16 bytes to lds + 16 lane (lds wave-uniform).
__device__ __forceinline__ void store16(uint8_t* lds, u4 v) {
  *reinterpret_cast<u4*>(lds + (threadIdx.x & 63u) * 16) = v;
}

// 16 bytes per lane into lds + 16 lane (lds wave-uniform). Dma: the direct
// copy, from 16-byte aligned sources. Otherwise through registers, from
// sources of any alignment.
template <bool Dma>
__device__ __forceinline__ void copy16(const uint8_t* g, uint8_t* lds) {
  if constexpr (Dma)
    __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
  else
    store16(lds, load16(g));
}

// c ? a : b by value. (The operator on variables that a lambda captured by
// reference selects their addresses, and they then live in scratch.)
__device__ __forceinline__ const uint8_t* pick(bool c, const uint8_t* a, const uint8_t* b) { return c ? a : b; }

// FP32 at a 16-byte aligned address, or at any.
template <bool Aligned>
__device__ __forceinline__ float load_f32(const uint8_t* p) {
  if constexpr (Aligned) return *reinterpret_cast<const float*>(p);
  return __uint_as_float(uint32_t(p[0]) | uint32_t(p[1]) << 8 | uint32_t(p[2]) << 16 | uint32_t(p[3]) << 24);
}

// Calls f with the ring's slots (and a table beside them) as pairwise disjoint __restrict__ pointers, so
// that the compiler adds no wait for the copies in flight into one slot before
// the reads of another (the ring's own waits are explicit).
template <class F>
__device__ __attribute__((always_inline)) inline void with_slots(uint8_t* __restrict__ s0, uint8_t* __restrict__ s1,
                                                                 uint8_t* __restrict__ s2, uint8_t* __restrict__ s3,
                                                                 uint8_t* __restrict__ table, F&& f) {
  f(s0, s1, s2, s3, table);
}

// The ring over `count` chunks: start(c, slot) for the first NS - 1, then
// step(c, slot) in order, slot = c % NS as a compile-time constant (which is
// what keeps the slots' pointers apart in with_slots).
template <int NS, class Start, class Step>
__device__ __attribute__((always_inline)) inline void ring(uint32_t count, Start&& start, Step&& step) {
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;
  start(0u, C0{});
  if constexpr (NS > 2) start(1u, C1{});
  if constexpr (NS > 3) start(2u, C2{});
  for (uint32_t c = 0; c < count; c += NS) {
    step(c, C0{});
    if (c + 1 < count) step(c + 1, C1{});
    if constexpr (NS > 2)
      if (c + 2 < count) step(c + 2, C2{});
    if constexpr (NS > 3)
      if (c + 3 < count) step(c + 3, C3{});
  }
}

// Tile of a block: WR x WT waves, each NI x NJ MFMA tiles (16 weight rows x 16
// tokens); NS ring slots of one K chunk.
//
// Weight rows. The block's BR LDS rows are `Halves` equal parts (two for a
// gate / up pair: gate rows first, then the up rows of the same features) and
// a wave owns 16 H consecutive rows of each part (H = NI / Halves). MFMA row a
// of the wave's tile i is part i / H, row 4 H (a / 4) + 4 (i % H) + a % 4 of
// those 16 H: the four results of a lane and its H tiles are then 4 H
// consecutive rows of one token, which store as one run.
template <int WR_, int WT_, int NI_, int NJ_, int NS_, bool Paired_>
struct Tile {
  static constexpr int WR = WR_, WT = WT_, NI = NI_, NJ = NJ_, NS = NS_;
  static constexpr bool Paired = Paired_;
  static constexpr int Halves = Paired ? 2 : 1, H = NI / Halves;
  static_assert(NI % Halves == 0 && NS >= 2 && NS <= 4, "tile");
  static constexpr uint32_t W = WR * WT, BR = 16 * WR * NI, BT = 16 * WT * NJ, HR = BR / Halves;
  static constexpr uint32_t Units = (BR + BT) / 8;             // 8-row copies of 1 KB per chunk
  static constexpr uint32_t PerWave = (Units + W - 1) / W;     // the last ones repeat unit Units - 1
  static constexpr uint32_t RowBytes = (BR + BT) * 128;

  // LDS row of (wave row wr, tile i, MFMA row a)
  static __host__ __device__ constexpr uint32_t row(uint32_t wr, int i, uint32_t a) {
    return (i / H) * HR + wr * (16 * H) + (a >> 2) * (4 * H) + (i % H) * 4 + (a & 3u);
  }
  // XOR keys of weight row R and token row t (the inverse of row() gives a)
  static __host__ __device__ constexpr uint32_t key_w(uint32_t R) {
    const uint32_t l = R % (16 * H);
    return ((l & 3u) >> 1) | ((l / (4 * H)) << 1);
  }
  static __host__ __device__ constexpr uint32_t key_a(uint32_t a) { return a >> 1; }
  static __host__ __device__ constexpr uint32_t key_t(uint32_t t) { return (t >> 1) & 7u; }
};

// A tile's rows and tokens, the blocks of it that share a CU, and the time of
// a K chunk with 1 .. share of them on it.
struct TileCost {
  uint32_t rows, toks, share;
  float t[8];
};

// The tile whose busiest of `cus` CUs finishes an rows x toks grid first: its
// index, and that time per K chunk.
struct TilePick {
  uint32_t index;
  float time;
};

template <class Costs>
inline TilePick pick_tile(const Costs& c, uint64_t rows, uint64_t toks, uint32_t cus) {
  TilePick best{0, 0.f};
  for (uint32_t i = 0; i < std::size(c); ++i) {
    const uint64_t blocks = (rows + c[i].rows - 1) / c[i].rows * ((toks + c[i].toks - 1) / c[i].toks);
    const uint64_t b = (blocks + cus - 1) / cus, rest = b % c[i].share;
    const float t = float(b / c[i].share) * c[i].t[c[i].share - 1] + (rest ? c[i].t[rest - 1] : 0.f);
    if (i == 0 || t < best.time) best = {i, t};
  }
  return best;
}

inline bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Tile index of a block: consecutive tiles go to one XCD (blocks are dealt to
// the eight XCDs in turn), so blocks that share weight rows share its L2.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t nblk) {
  const uint32_t x = b % 8, q = nblk / 8, r = nblk % 8;
  return x * q + min(x, r) + b / 8;
}

// Stores one lane's run of N consecutive results of a token row as BF16. vec: y
// is 8-byte aligned.
template <int N>
__device__ __forceinline__ void store_bf16_run(uint16_t* y, const float (&v)[N], bool vec) {
  uint32_t w[N / 2];
#pragma unroll
  for (int e = 0; e < N / 2; ++e)
    w[e] = uint32_t(f32_to_bf16_rne(v[2 * e])) | (uint32_t(f32_to_bf16_rne(v[2 * e + 1])) << 16);
  if (vec) {
#pragma unroll
    for (int e = 0; e < N / 4; ++e) reinterpret_cast<uint2*>(y)[e] = make_uint2(w[2 * e], w[2 * e + 1]);
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) y[e] = uint16_t(w[e / 2] >> (16 * (e & 1)));
  }
}

}  // namespace qw38hip
