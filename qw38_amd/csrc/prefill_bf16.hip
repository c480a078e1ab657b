// BF16 prefill projection over Q4_K weights (layout 0x020D) on gfx950 matrix
// cores: Y[m][n] = X[m][k] (BF16) * W^T, W rebuilt as BF16 operands.
//
// Semantics (cuda/prefill.cu:62-77, 116-142, 510-715): every weight is the
// BF16 operand BF16_RNE(fl(fl(d * s_g) * c) - fl(dmin * m_g)) -- the same
// operand as the BF16 decode GEMV, built here with fma(ds, c, -dm), which is
// bit-identical because fl(d * s) * c is exact -- and the products with the
// BF16 activations are summed in FP32 (v_mfma_f32_16x16x32_bf16, the matrix
// core accumulating over all of K). Epilogues: StoreBf16, StoreFp32,
// ResidualAddFp32; the paired gate/up launch writes BF16(SiLU(g) * u).
//
// The raw 0x020D bytes and the activations are copied straight into LDS
// rings (no registers, no VALU work, one barrier per 64-wide K step), and each
// wave rebuilds the operands of its own rows in registers, once for all of
// the tile's tokens. What bounds it is the vector ALU: about 25 instructions
// per 16x16x32 operand fragment (17 to rebuild it, the rest scales and
// addresses), which run mostly beside and not under the matrix cores (at 112
// tokens per tile 3.6 per MFMA, the matrix cores 28 to 31% busy), and the LDS
// reads of the activation fragments (1 KB per MFMA and row tile pair). Two row
// tiles per wave halve those against one; four (128 tokens) do not fit 256
// VGPRs. Bank conflicts: none, but for 8 cycles per wave and step where the
// compiler joins the code reads of two row tiles.
//
// Before, 256 x 256 / 256 x 128 / 128 x 64 tiles rebuilt the operands into
// LDS; large grids of the biggest are fast (prefill_big_kernel), but every other
// shape waited out a load latency per step. Microseconds, before -> now, weights not cached:
//                       16       64      300      512     1024        4096 tokens
//   2 x 17408 x 5120   89>45  121>68  250>163  275>199  460>373  1621>1385
//   5120 x 17408      179>63  180>77  191>124  257>159  289>247    774>711
//   12288 x 5120       55>23   57>33   82>64    92>81   180>132    473>466
#include <array>

#include "lds_gemm.hpp"
#include "q4k_operands.hpp"

namespace qw38hip {
namespace {

typedef uint32_t u2 __attribute__((ext_vector_type(2)));

// Tile of a block: WR waves, each 16 NI weight rows x all BT = 16 NJ tokens.
// Weights (codes and metadata) are staged by super-block in NA slots,
// activations by 64-wide K step in NS slots.
template <int WR_, int NI_, int NJ_, int NS_, int NA_, bool Paired_>
struct RingTile {
  static constexpr int WR = WR_, NI = NI_, NJ = NJ_, NS = NS_, NA = NA_;
  static constexpr bool Paired = Paired_;
  static constexpr int Halves = Paired ? 2 : 1, H = NI / Halves;
  static_assert(NI % Halves == 0 && NS >= 2 && NA >= 2, "tile");
  static constexpr uint32_t W = WR, BR = 16 * WR * NI, BT = 16 * NJ, HR = BR / Halves;
  // 1 KB copies: an 8-row strip's codes; the metadata of eight strips of one
  // half; eight tokens' 64 activations
  static constexpr uint32_t UA = BR / 8, UMh = (HR + 63) / 64, UM = UMh * Halves, UB = BT / 8;
  // a quarter of a super-block's weight copies goes out with each K step
  static constexpr uint32_t Quarter = (UA + UM + 3) / 4;
  static constexpr uint32_t PA = (Quarter + W - 1) / W, PB = (UB + W - 1) / W;
  static constexpr uint32_t OffM = UA * 1024, SlotA = (UA + UM) * 1024, SlotB = UB * 1024, OffB = NA * SlotA;
  static constexpr uint32_t Lds = OffB + NS * SlotB;
  static constexpr int Flight = (NS - 2) * int(PA + PB);
  // at a super-block's first step its last quarter, one step old when NA = 2, has landed too
  static constexpr int Flight0 = NA == 2 && int(PB) < Flight ? int(PB) : Flight;
  static_assert(NA == 2 || NS <= 4 * NA - 6, "a super-block's copies land before its first step");

  static __host__ __device__ constexpr uint32_t row(uint32_t wr, int i, uint32_t a) {
    return (i / H) * HR + wr * (16 * H) + (a >> 2) * (4 * H) + (i % H) * 4 + (a & 3u);
  }
  static __host__ __device__ constexpr uint32_t key_w(uint32_t R) {
    const uint32_t l = R % (16 * H);
    return ((l & 3u) >> 1) | ((l / (4 * H)) << 1);
  }
  // Token rows: pieces 2 lk + s of lanes lk, lk + 1 meet in one group of a b128
  // read ({0-3, 12-15, 20-23, 24-27}), so pairs of rows that differ in bit 1 of
  // t / 2 must not differ in that bit of the key alone.
  static __host__ __device__ constexpr uint32_t key_t(uint32_t t) {
    const uint32_t a = (t >> 1) & 7u;
    return a ^ ((a & 2u) << 1);
  }
  // Metadata of row R of a half stands at meta_at(R): a fragment's 16 rows side by side.
  static __host__ __device__ constexpr uint32_t meta_at(uint32_t R) {
    const uint32_t l = R % (16 * H);
    return R - l + (l / 4 % H) * 16 + l / (4 * H) * 4 + l % 4;
  }
  static __host__ __device__ constexpr uint32_t meta_row(uint32_t at) {  // its inverse
    const uint32_t l = at % (16 * H);
    return at - l + (l % 16 / 4) * (4 * H) + l / 16 * 4 + l % 4;
  }
};

__device__ __forceinline__ bool vector_rows(const void* out, const float* residual, uint32_t n) {
  return n % 4 == 0 && ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 15u) == 0;
}

// A lane's results of rows row .. row + 3 for one token (u: the up rows'),
// with `vec` as vectors. Whole: with `vec` the rows are known to be all below n
// or all past it.
template <bool Paired, bool Whole>
__device__ __forceinline__ void store_rows(void* out, const float* residual, int epi, bool vec, uint32_t n, uint32_t m,
                                           uint32_t row, uint32_t tok, f4 g, f4 u) {
  if (tok >= m || row >= n) return;
  const size_t o = size_t(tok) * n + row;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = Paired ? silu(g[e]) * u[e] : g[e];
  if ((Whole || row + 4 <= n) && vec) {
    if (Paired || epi == QW38_DECODE_STORE_BF16) {
      store_bf16_run<4>(static_cast<uint16_t*>(out) + o, v, true);
      return;
    }
    if (epi == QW38_DECODE_RESIDUAL_ADD_FP32) {
      const float4 p = *reinterpret_cast<const float4*>(residual + o);
      v[0] = p.x + v[0];
      v[1] = p.y + v[1];
      v[2] = p.z + v[2];
      v[3] = p.w + v[3];
    }
    *reinterpret_cast<float4*>(static_cast<float*>(out) + o) = make_float4(v[0], v[1], v[2], v[3]);
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (row + e >= n) continue;
    if (Paired || epi == QW38_DECODE_STORE_BF16)
      static_cast<uint16_t*>(out)[o + e] = f32_to_bf16_rne(v[e]);
    else
      static_cast<float*>(out)[o + e] = epi == QW38_DECODE_STORE_FP32 ? v[e] : residual[o + e] + v[e];
  }
}

// The results of a wave whose lanes hold more than eight runs of rows: each(f)
// calls f(row, token, g, u) for them. The form is chosen once, outside of the runs:
// chosen at every run, the skipped code of the other forms costs a launch 1.5 us
// (65536 x 256 at 150 tokens: 17.8 -> 16.5 us). With fewer runs it gains nothing.
template <bool Paired, class Each>
__device__ __forceinline__ void store_tile(void* out, const float* residual, int epi, uint32_t n, uint32_t m,
                                           Each&& each) {
  const bool vec = vector_rows(out, residual, n);
  auto all = [&](int e, bool v) __attribute__((always_inline)) {
    each([&](uint32_t row, uint32_t tok, f4 g, f4 u) __attribute__((always_inline)) {
      store_rows<Paired, true>(out, residual, e, v, n, m, row, tok, g, u);
    });
  };
  if (!vec) all(epi, false);
  else if (Paired || epi == QW38_DECODE_STORE_BF16) all(QW38_DECODE_STORE_BF16, true);
  else if (epi == QW38_DECODE_STORE_FP32) all(QW38_DECODE_STORE_FP32, true);
  else all(QW38_DECODE_RESIDUAL_ADD_FP32, true);
}

template <class T, bool Dma>
__global__ __launch_bounds__(T::W * 64, 2) void prefill_kernel(
    const uint8_t* __restrict__ codes_a, const uint8_t* __restrict__ meta_a, const uint8_t* __restrict__ codes_b,
    const uint8_t* __restrict__ meta_b, uint32_t n, uint32_t k, const uint16_t* __restrict__ x, uint32_t m, void* out,
    const float* __restrict__ residual, int epi, uint32_t tok_blocks, uint32_t row_base) {
  constexpr int NI = T::NI, NJ = T::NJ, NS = T::NS, NA = T::NA, H = T::H;
  static_assert(b128_clean([](uint32_t l) { return l % 16 * 128 + ((l / 16 * 2) ^ T::key_t(l % 16)) * 16; }) &&
                    b128_clean([](uint32_t l) { return T::meta_at(T::row(0, 0, l % 16)) * 16; }),
                "fragment and metadata reads");
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t row0 = row_base + tile / tok_blocks * T::HR, tok0 = tile % tok_blocks * T::BT;
  const uint32_t lane = threadIdx.x & 63u, wr = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lr = lane & 15u, lk = lane >> 4;
  const uint32_t kbs = k / 256;

  // Copies of strips past the last re-read it, of tokens past m the last token.
  const uint32_t strips = (n + 7) / 8, strip0 = row0 / 8;
  const uint8_t* const ca = codes_a + uint64_t(strip0) * kbs * 1024;
  const uint8_t* const ma = meta_a + uint64_t(strip0) * kbs * 128;
  const uint8_t* const cb = T::Paired ? codes_b + uint64_t(strip0) * kbs * 1024 : ca;
  const uint8_t* const mb = T::Paired ? meta_b + uint64_t(strip0) * kbs * 128 : ma;
  const uint32_t last = strips - 1 - strip0;
  auto each_a = [&](uint32_t kb_in, uint32_t q, uint8_t* slot, auto&& f) __attribute__((always_inline)) {
    const uint32_t kb = min(kb_in, kbs - 1);
#pragma unroll
    for (uint32_t u = 0; u < T::PA; ++u) {
      const uint32_t unit = min(q * T::Quarter + wr + u * T::W, T::UA + T::UM - 1);  // wave-uniform
      const uint8_t* src;
      if (unit < T::UA) {
        const uint32_t st = min(unit % (T::HR / 8), last);
        src = pick(unit >= T::HR / 8, cb, ca) + uint64_t(st * kbs + kb) * 1024 +
              ((lane >> 3) * 128 + ((lane & 7u) ^ T::key_w(unit * 8 + (lane >> 3))) * 16);
      } else {
        const uint32_t v = unit - T::UA, R = T::meta_row(v % T::UMh * 64 + lane), st = min(R / 8, last);
        src = pick(v >= T::UMh, mb, ma) + (st * kbs + kb) * 128 + R % 8 * 16;
      }
      f(src, slot + unit * 1024, u);
    }
  };
  uint32_t toff[T::PB];
#pragma unroll
  for (uint32_t u = 0; u < T::PB; ++u) {
    const uint32_t t = min(wr + u * T::W, T::UB - 1) * 8 + (lane >> 3);
    toff[u] = min(tok0 + t, m - 1) * (2 * k) + ((lane & 7u) ^ T::key_t(t)) * 16;
  }
  auto each_b = [&](uint32_t c_in, uint8_t* slot, auto&& f) __attribute__((always_inline)) {
    const uint8_t* base = reinterpret_cast<const uint8_t*>(x) + min(c_in, 4 * kbs - 1) * 128;
#pragma unroll
    for (uint32_t u = 0; u < T::PB; ++u) f(base + toff[u], slot + min(wr + u * T::W, T::UB - 1) * 1024, u);
  };
  auto copy = [&](const uint8_t* src, uint8_t* dst, uint32_t) __attribute__((always_inline)) { copy16<Dma>(src, dst); };
  // Without direct copies a step's share is loaded to registers one step
  // before it is stored, so that no wave waits out the load latency.
  u4 ra[Dma ? 1 : T::PA], rb[Dma ? 1 : T::PB];
  auto load = [&](uint32_t kb, uint32_t q, uint32_t c) __attribute__((always_inline)) {
    each_a(kb, q, nullptr, [&](const uint8_t* src, uint8_t*, uint32_t u) __attribute__((always_inline)) { ra[u] = load16(src); });
    each_b(c, nullptr, [&](const uint8_t* src, uint8_t*, uint32_t u) __attribute__((always_inline)) { rb[u] = load16(src); });
  };

  f4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f4{0, 0, 0, 0};

  // Lane (lr, lk) holds 16 codes, half lk % 2 of group 2 q + lk / 2, of each
  // row tile's row lr, and the matching 16 activations of each token tile's
  // token lr: two MFMAs.
  auto compute = [&](auto qc, const uint8_t* sa, const uint8_t* sb) __attribute__((always_inline)) {
    constexpr uint32_t q = decltype(qc)::value;
    u2 w[NI];
    float ds24[NI], ds20[NI], ndm[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t R = T::row(wr, i, lr);
      w[i] = *reinterpret_cast<const u2*>(sa + R * 128 + (((2 * q + (lk >> 1)) ^ (lr >> 1)) * 16) + (lk & 1u) * 8);
      const u4 mt = *reinterpret_cast<const u4*>(sa + T::OffM + (i / H) * (T::UMh * 1024) + T::meta_at(R % T::HR) * 16);
      const uint32_t sh = 8u * ((2 * q + (lk >> 1)) & 3u);
      uint32_t sc, mn;
      if constexpr (q < 2) {
        sc = __builtin_amdgcn_ubfe(mt.y, sh, 6u);
        mn = __builtin_amdgcn_ubfe(mt.z, sh, 6u);
      } else {
        sc = __builtin_amdgcn_ubfe(mt.w, sh, 4u) | (__builtin_amdgcn_ubfe(mt.y, sh + 6u, 2u) << 4);
        mn = __builtin_amdgcn_ubfe(mt.w, sh + 4u, 4u) | (__builtin_amdgcn_ubfe(mt.z, sh + 6u, 2u) << 4);
      }
      const float ds = f16_to_f32(mt.x & 0xffffu) * float(sc);  // exact
      ndm[i] = -(f16_to_f32(mt.x >> 16) * float(mn));           // exact
      ds24[i] = ds * 0x1p24f;
      ds20[i] = ds * 0x1p20f;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf8 af[NI];
#pragma unroll
      for (int i = 0; i < NI; ++i) af[i] = operands8(w[i][s], ds24[i], ds20[i], ndm[i]);
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const bf8 bf = *reinterpret_cast<const bf8*>(sb + (j * 16 + lr) * 128 + ((2 * lk + s) ^ T::key_t(lr)) * 16);
#pragma unroll
        for (int i = 0; i < NI; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf, acc[i][j], 0, 0, 0);
      }
    }
  };

  // Step c = 4 kb + q awaits its copies (the NS - 2 younger steps' may stay in
  // flight); the barrier publishes them and retires step c - 1 (at q = 0 also
  // super-block kb - 1), whose slot takes step c + NS - 1 (quarter q of
  // super-block kb + NA - 1). Copies past the end re-read the last data into
  // retired slots.
  uint32_t cur = 0, nxt = (NS - 1) * T::SlotB, acur = 0, anxt = (NA - 1) * T::SlotA;
  auto step = [&](auto qc, uint32_t kb) __attribute__((always_inline)) {
    constexpr uint32_t q = decltype(qc)::value;
    copies_barrier<!Dma ? 63 : q == 0 ? T::Flight0 : T::Flight>();
    if constexpr (Dma) {
      each_a(kb + NA - 1, q, lds + anxt, copy);
      each_b(4 * kb + q + NS - 1, lds + T::OffB + nxt, copy);
    } else {
      each_a(kb + NA - 1, q, lds + anxt,
             [&](const uint8_t*, uint8_t* dst, uint32_t u) __attribute__((always_inline)) { store16(dst, ra[u]); });
      each_b(4 * kb + q + NS - 1, lds + T::OffB + nxt,
             [&](const uint8_t*, uint8_t* dst, uint32_t u) __attribute__((always_inline)) { store16(dst, rb[u]); });
      load(kb + NA - 1 + (q + 1) / 4, (q + 1) % 4, 4 * kb + q + NS);
    }
    __builtin_amdgcn_sched_barrier(0);  // the copies go out before the step's work
    compute(qc, lds + acur, lds + T::OffB + cur);
    nxt = cur;
    cur = cur + T::SlotB == NS * T::SlotB ? 0 : cur + T::SlotB;
  };
#pragma unroll
  for (int s = 0; s < NA - 1; ++s)
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) each_a(s, q, lds + s * T::SlotA, copy);
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) each_b(s, lds + T::OffB + s * T::SlotB, copy);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the steady state's counts hold from step 0 on
  if constexpr (!Dma) load(NA - 1, 0, NS - 1);
  for (uint32_t kb = 0; kb < kbs; ++kb) {
    step(std::integral_constant<uint32_t, 0>{}, kb);
    step(std::integral_constant<uint32_t, 1>{}, kb);
    step(std::integral_constant<uint32_t, 2>{}, kb);
    step(std::integral_constant<uint32_t, 3>{}, kb);
    anxt = acur;
    acur = acur + T::SlotA == NA * T::SlotA ? 0 : acur + T::SlotA;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy outlives the block

  const uint32_t r = row0 + wr * (16 * H) + lk * (4 * H);
  if constexpr (H * NJ > 8) {
    store_tile<T::Paired>(out, residual, epi, n, m, [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < H; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) f(r + 4 * i, tok0 + j * 16 + lr, acc[i][j], acc[NI - H + i][j]);
    });
  } else {
    const bool vec = vector_rows(out, residual, n);
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        store_rows<T::Paired, false>(out, residual, epi, vec, n, m, r + 4 * i, tok0 + j * 16 + lr, acc[i][j],
                                     acc[NI - H + i][j]);
  }
}

// 256 x 256 tile for large grids: eight waves of 64 x 128, one
// block per CU. Threads rebuild the operands of a K step into LDS for all
// waves, so a weight is rebuilt once per 256 tokens, and the wave tiles read
// half the activation fragments per MFMA of the ring tiles (whose waves hold 32
// rows). The second wave of each SIMD runs its MFMAs before its staging.
// Paired: the rows are 128 features of the gate and of the up weight, and a
// wave holds both of its 32 features.
//
// Which K index an MFMA slot holds is as in prefill_kernel, so both give the
// same bits: lane (lr, lk) takes piece 2 lk + h (eight K indexes) in MFMA h. A
// row is 160 B of LDS with that piece at position 4 h + gray(lk): a b128
// access is served in lane groups like {0-3, 12-15, 20-23, 24-27}, and both the
// fragment reads (rows lr, pairs of neighbouring lk) and the staging stores (rows
// of lane / 2, pieces of the two K32 halves) then hit 16 distinct 16-byte slots.
constexpr int kBigStride = 80;
__host__ __device__ constexpr uint32_t big_piece(uint32_t p) {  // offset in halfs
  const uint32_t lk = p >> 1;
  return ((p & 1u) * 4 + (lk ^ (lk >> 1))) * 8;
}

template <bool Paired, int BT>
__global__ __launch_bounds__(512, 1) void prefill_big_kernel(
    const uint8_t* __restrict__ codes_a, const uint8_t* __restrict__ meta_a, const uint8_t* __restrict__ codes_b,
    const uint8_t* __restrict__ meta_b, uint32_t n, uint32_t k, const uint16_t* __restrict__ x, uint32_t m, void* out,
    const float* __restrict__ residual, int epi, uint32_t tok_blocks, uint32_t row_base) {
  constexpr int BR = 256, NJ = BT / 32, HR = Paired ? BR / 2 : BR, XP = BT / 64;
  static_assert(b128_clean([](uint32_t l) { return (l % 16 * kBigStride + big_piece(l / 16 * 2)) * 2; }) &&
                    b128_clean([](uint32_t l) { return (l / 2 * kBigStride + big_piece(l % 2 * 4)) * 2; }),
                "fragment reads, staging stores");
  __shared__ __align__(16) uint16_t a_lds[2][BR * kBigStride];
  __shared__ __align__(16) uint16_t b_lds[2][BT * kBigStride];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t row0 = row_base + tile / tok_blocks * HR, tok0 = tile % tok_blocks * BT;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t wr = wave >> 1, wt = wave & 1u, lr = lane & 15u, lk = lane >> 4;
  const uint32_t kbs = k / 256, steps = k / 64;

  // thread: row ar's K32 group asel, and XP pieces of token bt's 64 inputs. Paired:
  // rows 0..127 are gate rows, 128..255 the up rows of the same features.
  const uint32_t ar = tid >> 1, asel = tid & 1u, bt = tid * XP / 8, bp = tid * XP % 8;
  const bool up = Paired && __builtin_amdgcn_readfirstlane(tid) >= 256;
  const uint8_t* const codes = pick(up, codes_b, codes_a);
  const uint8_t* const meta = pick(up, meta_b, meta_a);
  const uint32_t arow = min(row0 + ar % HR, (n + 7) / 8 * 8 - 1);
  const uint64_t trow0 = uint64_t(arow / 8) * kbs * 8 + arow % 8;
  const uint16_t* xrow = x + size_t(min(tok0 + bt, m - 1)) * k + bp * 8;
  // LDS row of the wave's tile i: four row tiles, or two gate and their two up tiles
  const auto arow_lds = [&](int i) __attribute__((always_inline)) {
    return Paired ? (i >> 1) * HR + wr * 32 + (i & 1) * 16 + lr : wr * 64 + i * 16 + lr;
  };

  f4 acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f4{0, 0, 0, 0};

  u4 fc, fm, xv[XP];
  auto fetch = [&](uint32_t s) __attribute__((always_inline)) {
    const uint64_t tr = trow0 + (s >> 2) * 8;
    fc = load16(codes + tr * 128 + (2 * (s & 3u) + asel) * 16);
    fm = load16(meta + tr * 16);
#pragma unroll
    for (int q = 0; q < XP; ++q) xv[q] = load16(reinterpret_cast<const uint8_t*>(xrow + s * 64 + 8 * q));
  };
  auto stage = [&](uint32_t s) __attribute__((always_inline)) {
    float sc, mn;
    q4_scale_min_lane(fm.y, fm.z, fm.w, 2 * (s & 3u) + asel, sc, mn);
    const float ds = f16_to_f32(fm.x & 0xffffu) * sc;      // exact
    const float ndm = -(f16_to_f32(fm.x >> 16) * mn);      // exact
    uint16_t* da = &a_lds[s & 1u][ar * kBigStride];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<bf8*>(da + big_piece(4 * asel + q)) = operands8(fc[q], ds * 0x1p24f, ds * 0x1p20f, ndm);
    uint16_t* db = &b_lds[s & 1u][bt * kBigStride];
#pragma unroll
    for (int q = 0; q < XP; ++q) *reinterpret_cast<u4*>(db + big_piece(bp + q)) = xv[q];
  };
  bf8 af[4], bf[NJ];
  auto frags = [&](uint32_t buf, int h) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      bf[j] = *reinterpret_cast<const bf8*>(&b_lds[buf][(wt * (BT / 2) + j * 16 + lr) * kBigStride + big_piece(2 * lk + h)]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      af[i] = *reinterpret_cast<const bf8*>(&a_lds[buf][arow_lds(i) * kBigStride + big_piece(2 * lk + h)]);
  };
  auto mma = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
  };

  fetch(0);
  stage(0);
  if (steps > 1) fetch(1);
  // The time of a step depends on where the loop lies in the 32-byte windows of
  // the instruction fetch, where the grid leaves the chip the power for it: 129 to
  // 135 us over the eight places (17408 x 5120 at 512 tokens), paired 135 to 146 (5120
  // features at 1024). These are the best places.
  asm volatile(".p2align 5\n\t.rept %0\n\ts_nop 0\n\t.endr" ::"n"(Paired ? 5 : 4));
  for (uint32_t s = 0; s < steps; ++s) {
    __syncthreads();
    const uint32_t buf = s & 1u;
    frags(buf, 0);
    if (wave >= 4) {
      __builtin_amdgcn_s_setprio(1);
      mma();
      frags(buf, 1);
      mma();
      __builtin_amdgcn_s_setprio(0);
      if (s + 1 < steps) stage(s + 1);
      if (s + 2 < steps) fetch(s + 2);
    } else {
      if (s + 1 < steps) stage(s + 1);
      if (s + 2 < steps) fetch(s + 2);
      __builtin_amdgcn_s_setprio(1);
      mma();
      frags(buf, 1);
      mma();
      __builtin_amdgcn_s_setprio(0);
    }
  }

  constexpr int H = Paired ? 2 : 4;
  store_tile<Paired>(out, residual, epi, n, m, [&](auto&& f) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < H; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        f(row0 + (wr * H + i) * 16 + lk * 4, tok0 + wt * (BT / 2) + j * 16 + lr, acc[i][j], acc[4 - H + i][j]);
  });
}

}  // namespace

namespace {
struct PrefillArgs {
  const WeightView *a, *b;
  const uint16_t* x;
  uint32_t m;
  void* out;
  const float* residual;
  int epilogue;
  hipStream_t s;
  uint32_t row_base;
};

template <class T, bool Dma>
hipError_t prefill_tile(const PrefillArgs& p) {
  const hipError_t e = set_max_lds(reinterpret_cast<const void*>(&prefill_kernel<T, Dma>), T::Lds);
  if (e != hipSuccess) return e;
  const uint32_t tb = (p.m + T::BT - 1) / T::BT;
  hipLaunchKernelGGL((prefill_kernel<T, Dma>), dim3((p.a->n - p.row_base + T::HR - 1) / T::HR * tb), dim3(T::W * 64), T::Lds, p.s,
                     p.a->codes, p.a->scales, p.b ? p.b->codes : nullptr, p.b ? p.b->scales : nullptr, p.a->n, p.a->k,
                     p.x, p.m, p.out, p.residual, p.epilogue, tb, p.row_base);
  return hipGetLastError();
}

// row_blocks blocks of 256 x BT tiles from row p.row_base on.
template <bool P, int BT>
hipError_t prefill_big(const PrefillArgs& p, uint32_t row_blocks) {
  const uint32_t tb = (p.m + BT - 1) / BT;
  hipLaunchKernelGGL((prefill_big_kernel<P, BT>), dim3(row_blocks * tb), dim3(512), 0, p.s, p.a->codes, p.a->scales,
                     p.b ? p.b->codes : nullptr, p.b ? p.b->scales : nullptr, p.a->n, p.a->k, p.x, p.m, p.out,
                     p.residual, p.epilogue, tb, p.row_base);
  return hipGetLastError();
}

// Ring tiles by the busiest CU's time per 64-wide K step, in microseconds with
// one, two, ... blocks on it, measured at K = 5120 and 17408 (1024 to 65536
// rows, 16 to 4096 tokens), and a round of big tiles. All tiles chain the same
// MFMAs over K in the same order, so the choice never changes a bit. Over 135 sizes
// (1024 to 34816 rows, 2 to 4096 tokens, K = 5120) it takes 0.6% longer than the best
// on average and at most 6%, gate/up pairs 2% and 14% (8704 features at 8 and 64
// tokens: 44 and 59 us, 39 and 51 on the 128 x 32 tile).
// Without direct copies a ring tile takes about 1.2 times as long (its share goes
// through registers and LDS stores), and a 256 x 128 big tile, which stages
// through registers anyway, takes the place of the 256 x 112 ring tile (12288 x
// 5120 at 512 tokens: 84 us against 97).
template <bool P>
constexpr auto tile_costs(bool dma) {
  auto c = [] {
    if constexpr (P)
      return std::array<TileCost, 6>{{{128, 128, 2, {0.78f, 1.2f}}, {256, 112, 1, {1.0f}},
                                      {128, 80, 2, {0.62f, 0.86f}}, {128, 64, 3, {0.59f, 0.74f, 1.02f}},
                                      {128, 32, 3, {0.45f, 0.59f, 0.81f}}, {64, 16, 3, {0.3f, 0.4f, 0.52f}}}};
    else
      return std::array<TileCost, 8>{{{128, 128, 2, {0.78f, 1.15f}}, {256, 112, 1, {0.98f}},
                                      {64, 128, 3, {0.65f, 0.73f, 1.03f}}, {128, 64, 3, {0.59f, 0.73f, 1.03f}},
                                      {64, 64, 3, {0.41f, 0.48f, 0.62f}}, {32, 32, 3, {0.34f, 0.37f, 0.4f}},
                                      {32, 16, 8, {0.235f, 0.29f, 0.305f, 0.36f, 0.41f, 0.49f, 0.57f, 0.65f}},
                                      {16, 16, 3, {0.24f, 0.245f, 0.265f}}}};
  }();
  if (!dma) {
    for (TileCost& tile : c)
      for (float& t : tile.t) t *= 1.2f;
    c[1] = {256, 128, 1, {P ? 1.1f : 1.02f}};
  }
  return c;
}

// Big tiles (256 tokens) on all rows, or on the rows of whole rounds with a ring
// tile behind, where that costs less than a ring tile alone. A full round takes
// 1.9 us per K step (paired 1.95), a partly filled one from 1.3 on. Ring tiles
// alone and with big ones, us: 17408 x 5120 at 768 tokens 167 and 148, 5120 x
// 17408 at 3072 637 and 484, 34816 x 5120 at 512 235 and 204; paired 17408
// features at 1024 425 and 391, at 4096 1716 and 1505. Two launches for less than 1%
// cost more than one (248320 x 2048 at 150 tokens: 265 and 254).
template <bool P>
GemmPlan prefill_plan(uint32_t n, uint32_t m, bool dma, uint32_t cus) {
  constexpr uint32_t hr = P ? 128 : 256;
  const auto costs = tile_costs<P>(dma);
  auto ring = [&](uint32_t rows) { return pick_tile(costs, uint64_t(rows) * (P ? 2 : 1), m, cus); };
  const uint32_t tb = (m + 255) / 256, all = (n + hr - 1) / hr;
  auto big = [&](uint32_t rb) {
    constexpr float full = P ? 1.95f : 1.9f, part = 1.3f;
    const uint64_t blocks = uint64_t(rb) * tb, rest = blocks % cus;
    return float(blocks / cus) * full + (rest ? part + (full - part) * float(rest) / float(cus) : 0.f);
  };
  const TilePick alone = ring(n);
  GemmPlan best{0, alone.index, uint32_t(costs.size())};
  float time = alone.time;
  if (big(all) < time) {
    best = {all, 0, best.tiles};
    time = big(all);
  }
  const uint32_t whole = uint32_t(uint64_t(n / hr) * tb / cus * cus / tb);
  if (whole > 0 && whole * hr < n) {
    const TilePick behind = ring(n - whole * hr);
    if (big(whole) + behind.time < 0.99f * time) best = {whole, behind.index, best.tiles};
  }
  return best;
}

template <bool P, bool Dma>
hipError_t prefill_run(PrefillArgs p) {
  constexpr uint32_t hr = P ? 128 : 256;
  const GemmPlan plan = prefill_plan<P>(p.a->n, p.m, Dma, uint32_t(cu_count()));
  if (plan.big) {
    const hipError_t e = prefill_big<P, 256>(p, plan.big);
    if (e != hipSuccess || plan.big * hr >= p.a->n) return e;
    p.row_base = plan.big * hr;
  }
#define QW38_PF(...) return prefill_tile<RingTile<__VA_ARGS__, P>, Dma>(p)
  switch (plan.tile) {
    case 0: QW38_PF(4, 2, 8, 2, 2);
    case 1:
      // A single super-block: the ring would be filled for it alone (65536 x 256 at 100
      // tokens: 13.3 us, 12.1 on the big tile; at K = 512 17.9 and 17.3, at 1024 25.9 and 26.9).
      if constexpr (Dma)
        if (P || p.a->k > 256) QW38_PF(8, 2, 7, 2, 2);
      return prefill_big<P, 128>(p, (p.a->n - p.row_base + hr - 1) / hr);
    case 2:
      if constexpr (P) QW38_PF(4, 2, 5, 2, 2);
      else QW38_PF(4, 1, 8, 2, 2);
    case 3: QW38_PF(4, 2, 4, 2, 2);
    case 4:
      if constexpr (P) QW38_PF(4, 2, 2, 4, 2);
      else QW38_PF(4, 1, 4, 3, 2);
    case 5:
      if constexpr (P) QW38_PF(2, 2, 1, 6, 3);
      else QW38_PF(2, 1, 2, 6, 4);
    case 6:
      if constexpr (!P) QW38_PF(2, 1, 1, 4, 2);
    default:
      if constexpr (!P) QW38_PF(1, 1, 1, 12, 6);
      else return hipErrorInvalidValue;
  }
#undef QW38_PF
}
}  // namespace

GemmPlan prefill_bf16_plan(bool paired, bool aligned, uint32_t n, uint32_t m, uint32_t cus) {
  return paired ? prefill_plan<true>(n, m, aligned, cus) : prefill_plan<false>(n, m, aligned, cus);
}

hipError_t launch_prefill_bf16(const WeightView& a, const WeightView* b, const uint16_t* x,
                               uint32_t m, void* out, const float* residual, int epilogue,
                               hipStream_t s) {
  if (a.layout != QW38_LAYOUT_Q4K_CANDIDATE_V2 || a.pk != a.k) return hipErrorInvalidValue;
  const PrefillArgs p{&a, b, x, m, out, residual, epilogue, s, 0};
  const bool dma = aligned16(a.codes) && aligned16(a.scales) && aligned16(x) &&
                   (!b || (aligned16(b->codes) && aligned16(b->scales)));
  if (b) return dma ? prefill_run<true, true>(p) : prefill_run<true, false>(p);
  return dma ? prefill_run<false, true>(p) : prefill_run<false, false>(p);
}

}  // namespace qw38hip
