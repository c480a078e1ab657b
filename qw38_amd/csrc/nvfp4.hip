// NVFP4 path of qw38's prefill and decode (cuda/nvfp4.hpp, cuda/nvfp4.cu,
// cuda/nvfp4_device.cuh, decode_mmv layout 0x020E):
//   pack_nvfp4   BF16 [m][k] -> E2M1 nibbles [m][pk/2] (element 2j in the low
//                nibble of byte j) + UE4M3 block scales of 16 elements in the
//                CUTLASS SM1xx swizzle over 128-row stripes (pad128(m) rows,
//                padding rows' scales 0, padding rows' codes not written);
//   weights      the same element/scale encoding of values / factor, where
//                factor is an FP32 power of two stored in bytes 0..3 of a
//                256-byte header in front of the scales
//                (src/compiler/quantization/nvfp4.cpp:25-56);
//   decode GEMV  BF16 x, weight element RN(RN(scale * factor) * value(code))
//                (cuda/decode_mmv.cu:94-102), FP32 FMAs, optional paired
//                SwiGLU, the decode_mmv epilogues;
//   W4A4 GEMM    y[t][r] = factor * sum_c (sa * a)(sw * w) (cuda/nvfp4.cu:
//                83-116), with the prefill epilogues fused into the store.
//
// The GEMM runs on FP16 MFMAs. gfx950's scaled FP4 MFMA and FP4 conversions
// take E8M0 (power-of-two) scales, and UE4M3 scales are not powers of two.
// But an E2M1 value times a UE4M3 value has at most 5 significant bits and
// lies in [2^-10, 2688], so it is exact in FP16: each operand fragment is
// converted exactly (v_cvt_scalef32_pk_f16_fp4 with scale 1, then a packed
// FP16 multiply by the block scale) and the MFMA chain runs over all of K
// without a per-block rescale. Products of two such FP16 values are exact in
// FP32, so the only rounding is the FP32 accumulation.
#include "lds_gemm.hpp"

namespace qw38hip {
namespace {

// ---- activation pack: eight elements per thread, two threads per 16-block;
// padding rows write only their scales (0). (Before, one thread
// per block loaded 2 bytes at a time and ran its 16 divides in turn.)
template <bool Vec>
__global__ __launch_bounds__(256) void pack_nvfp4_kernel(const uint16_t* __restrict__ x,
                                                         uint32_t m, uint32_t k, uint32_t pk,
                                                         uint8_t* __restrict__ codes,
                                                         uint8_t* __restrict__ scales) {
  const uint32_t per_row = pk / 8, t = blockIdx.x * 256 + threadIdx.x;  // the grid is whole rows of pad128(m)
  const uint32_t r = t / per_row, c = t % per_row * 8;
  const bool valid = r < m;
  float v[8];
  load8_bf16<Vec>(x + size_t(valid ? r : 0) * k, c, k, valid, v);
  uint32_t cw;
  const uint32_t s = nvfp4_encode_half(v, cw);
  if ((t & 1u) == 0) scales[nvfp4_sf_index(r, c / 16, pk)] = uint8_t(s);
  if (valid) *reinterpret_cast<uint32_t*>(codes + (size_t(r) * pk + c) / 2) = cw;
}

// ---- decode GEMV: 32 contiguous elements per lane and row ----
// Two consecutive 16-blocks per lane step; their scale bytes are adjacent in
// the swizzle (b even -> b % 4 in {0, 2}). A weight element is
// RN(RN(scale * factor) * value) (cuda/decode_mmv.cu:94-102): the UE4M3 scale
// has at most 4 significant bits and factor is a power of two, so
// scale * factor and its product with an E2M1 value (at most 2 significant
// bits) are exact in FP32. Each block is therefore summed as sum(value * x)
// with exact BF16 operands (v_cvt_scalef32_pk_bf16_fp4, then v_dot2_f32_bf16
// on element pairs) and scaled once: acc += (scale * factor) * block.
__device__ __forceinline__ float nvfp4_dot32(u4 c, uint32_t sf2, float factor,
                                             const uint32_t (&xw)[16], float acc) {
  typedef __bf16 bfx2 __attribute__((ext_vector_type(2)));
  const uint32_t cw[4] = {c[0], c[1], c[2], c[3]};
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const float sc = __fmul_rn(e4m3_value((sf2 >> (8 * h)) & 0xffu), factor);
    float bs = 0.f;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t word = cw[2 * h + w];
      const bfx2 v[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 0),
                         __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 1),
                         __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 2),
                         __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, 1.f, 3)};
#pragma unroll
      for (int bsel = 0; bsel < 4; ++bsel)
        bs = __builtin_amdgcn_fdot2_f32_bf16(v[bsel], __builtin_bit_cast(bfx2, xw[8 * h + 4 * w + bsel]), bs,
                                             false);
    }
    acc = fmaf(sc, bs, acc);
  }
  return acc;
}

__device__ __forceinline__ void decode_store(int epi, void* y, const float* residual, uint32_t row,
                                             float acc) {
  if (epi == QW38_DECODE_STORE_BF16) {
    static_cast<uint16_t*>(y)[row] = f32_to_bf16_rne(acc);
  } else if (epi == QW38_DECODE_RESIDUAL_ADD_FP32) {
    float* dst = y ? static_cast<float*>(y) : const_cast<float*>(residual);
    dst[row] = residual[row] + acc;
  } else {
    static_cast<float*>(y)[row] = acc;
  }
}

// A wave takes the rows r, r + 32, r + 64 and r + 96 of one 128-row stripe,
// whose scales for four blocks are the 16 bytes of one swizzle entry: one
// load per step fetches what four rows' separate loads would. Its steps (2048
// columns of the four rows; of the gate rows, then of the up rows) are loaded
// two ahead of the sums, behind the first of them the block stages x in LDS.
// Bound: HBM, and the FP4 conversions beside it. 2 x 17408 x 5120, weights not
// cached: 38.0 -> 26.6 us (3.8 TB/s), 17408 x 5120 19.2 -> 14.9, 5120 x 17408 22.5 ->
// 17.1, 1024 x 5120 6.5 -> 5.1. (Up to 512 rows of K = 512 it takes the 3.2 to 3.5 us
// of its launch, as the form before it did.)
struct GemvStep {
  u4 c[4];
  u4 s;
};

template <bool Paired>
__global__ __launch_bounds__(256) void nvfp4_gemv_kernel(
    const uint8_t* __restrict__ ca, const uint8_t* __restrict__ sa, const uint8_t* __restrict__ cb,
    const uint8_t* __restrict__ sb, uint32_t n, uint32_t pn, uint32_t k, uint32_t pk,
    const uint16_t* __restrict__ x, void* ya, void* yb, const float* ra, const float* rb, int epi) {
  constexpr uint32_t P = Paired ? 2 : 1;
  extern __shared__ __align__(16) uint8_t smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // 32 per stripe
  const uint32_t stripe = unit / 32, row0 = stripe * 128 + unit % 32;
  const uint32_t nsteps = (pk + 2047) / 2048, items = nsteps * P;

  // step i: columns 2048 (i % nsteps) + 32 lane of weight i / nsteps. Lanes
  // past pk load nothing and are not summed; rows past pn re-read
  // the last one and are not stored.
  uint32_t roff[4];
#pragma unroll
  for (uint32_t r = 0; r < 4; ++r) roff[r] = (min(row0 + 32 * r, pn - 1) - min(row0, pn - 1)) * (pk / 2);
  const size_t co = size_t(min(row0, pn - 1)) * (pk / 2);
  const size_t so = 256 + size_t(stripe) * 128 * (pk / 16) + (unit % 32) * 16;
  auto load = [&](uint32_t i, GemvStep& t) __attribute__((always_inline)) {
    const bool b = Paired && i >= nsteps;
    const uint32_t c = (b ? i - nsteps : i) * 2048 + lane * 32;
    if (c >= pk) return;
    const uint8_t* p = (b ? cb : ca) + co + c / 2;
#pragma unroll
    for (int r = 0; r < 4; ++r) t.c[r] = *reinterpret_cast<const u4*>(p + roff[r]);
    t.s = *reinterpret_cast<const u4*>((b ? sb : sa) + so + (c / 64) * 512);
  };
  const bool live = unit < (pn + 127) / 128 * 32 && row0 < pn;
  constexpr int D = 3;
  GemvStep st[D];
  if (live) {
#pragma unroll
    for (uint32_t i = 0; i < D; ++i)
      if (i < items) load(i, st[i]);
  }
  if ((reinterpret_cast<uintptr_t>(x) % 16) == 0 && k % 8 == 0) {
    for (uint32_t i = threadIdx.x; i < pk / 8; i += 256)
      reinterpret_cast<uint4*>(xs)[i] = 8 * i < k ? reinterpret_cast<const uint4*>(x)[i] : make_uint4(0, 0, 0, 0);
  } else {
    for (uint32_t i = threadIdx.x; i < pk; i += 256) xs[i] = i < k ? x[i] : uint16_t(0);
  }
  __syncthreads();
  if (!live) return;
  const float fa = *reinterpret_cast<const float*>(sa);
  const float fb = Paired ? *reinterpret_cast<const float*>(sb) : 0.f;
  float acc[P][4];
#pragma unroll
  for (uint32_t p = 0; p < P; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[p][r] = 0.f;
  auto sum = [&](uint32_t i, const GemvStep& t, float f, float (&a)[4]) __attribute__((always_inline)) {
    const uint32_t c = (i >= nsteps ? i - nsteps : i) * 2048 + lane * 32;
    if (c >= pk) return;
    uint32_t xw[16];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const u4 v = *reinterpret_cast<const u4*>(xs + c + 8 * q);
      xw[4 * q] = v.x; xw[4 * q + 1] = v.y; xw[4 * q + 2] = v.z; xw[4 * q + 3] = v.w;
    }
    const uint32_t sh = 16 * (lane & 1u);  // blocks 2 lane, 2 lane + 1 of the quad
#pragma unroll
    for (int r = 0; r < 4; ++r) a[r] = nvfp4_dot32(t.c[r], (t.s[r] >> sh) & 0xffffu, f, xw, a[r]);
  };
  for (uint32_t i = 0; i < items; i += D) {
#pragma unroll
    for (uint32_t u = 0; u < D; ++u) {
      if (i + u >= items) break;
      if (Paired && i + u >= nsteps) sum(i + u, st[u], fb, acc[P - 1]);
      else sum(i + u, st[u], fa, acc[0]);
      if (i + u + D < items) load(i + u + D, st[u]);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
      for (uint32_t p = 0; p < P; ++p) acc[p][r] += __shfl_xor(acc[p][r], o);
  if (lane != 0) return;
#pragma unroll
  for (uint32_t r = 0; r < 4; ++r) {
    const uint32_t row = row0 + 32 * r;
    if (row >= n) break;
    if (Paired && epi == QW38_DECODE_SWIGLU_BF16) {
      static_cast<uint16_t*>(ya)[row] = f32_to_bf16_rne(silu(acc[0][r]) * acc[P - 1][r]);
      continue;
    }
    decode_store(epi, ya, ra, row, acc[0][r]);
    if constexpr (Paired) decode_store(epi, yb, rb, row, acc[P - 1][r]);
  }
}

// ---- W4A4 GEMM ----
// fragment of the 16x16x32 f16 MFMA: 8 consecutive elements of one row,
// exact FP16 value * block scale
__device__ __forceinline__ half8 widen4(uint32_t w, _Float16 s) {
  const h2 ss{s, s};
  const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.f, 0) * ss;
  const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.f, 1) * ss;
  const h2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.f, 2) * ss;
  const h2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.f, 3) * ss;
  return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// One ring slot holds 256 elements of K: the raw codes (lds_gemm.hpp), then
// the swizzled block scales of the 128-row stripes that the tile's weight
// rows and tokens lie in, 2 KB each. A lane's 16-byte piece is 32 elements,
// two scale bytes side by side, and makes the fragments of four MFMAs.
template <class T>
struct Scales {
  static constexpr uint32_t PerPart = T::HR > 128 ? T::HR / 128 : 1, A = PerPart * T::Halves;
  static constexpr uint32_t B = T::BT > 128 ? T::BT / 128 : 1;
  static_assert((T::HR % 128 == 0 || 128 % T::HR == 0) && (T::BT % 128 == 0 || 128 % T::BT == 0), "stripes");
  static constexpr uint32_t Units = (A + B) * 2;  // 1 KB copies
  static constexpr uint32_t PerWave = (Units + T::W - 1) / T::W;
  static constexpr uint32_t Slot = T::RowBytes + Units * 1024;
  // byte of (row r of a stripe, element block b of the chunk's 16)
  static __device__ __forceinline__ uint32_t byte(uint32_t r, uint32_t b) {
    return (b / 4) * 512 + (r % 32) * 16 + (r / 32) * 4 + b % 4;
  }
};

// Operands: row-major nibbles (row stride pk / 2) and the swizzled UE4M3 of
// their 128-row stripes: wc / ws the weight (`rows` rows have codes), xc / xs
// the m tokens. epi 0 writes factor * sum as FP32 [m][n]; the decode epilogue
// IDs write the prefill epilogues (cuda/prefill.cu:116-134). Paired: wc is
// the gate and uc the up weight of the same n features, and the store is
// BF16(SiLU(gate) * up) (cuda/prefill.cu:203-215). `vec`: a BF16 output is
// 8-byte aligned (only qw38_prefill_mlp takes less; FP32 outputs and residuals
// are 16-byte aligned by the entries' checks).
//
// Bound: 6 VALU instructions per MFMA for widening both operands, and LDS: the
// scale bytes of a fragment's rows lie 16 bytes apart and share banks (56 cycles
// of conflicts per wave and chunk; the code fragments have none). Matrix cores
// 36% busy.
template <class T, bool Dma>
__global__ __launch_bounds__(T::W * 64) void nvfp4_gemm_kernel(
    const uint8_t* __restrict__ wc, const uint8_t* __restrict__ ws, const uint8_t* __restrict__ uc,
    const uint8_t* __restrict__ us, const uint8_t* fo, const uint8_t* fu, uint32_t n, uint32_t rows, uint32_t pk,
    const uint8_t* __restrict__ xc, const uint8_t* __restrict__ xs, uint32_t m, void* __restrict__ y,
    const float* __restrict__ residual, int epi, bool vec, uint32_t tok_blocks) {
  constexpr int NI = T::NI, NJ = T::NJ, NS = T::NS, H = T::H;
  using S = Scales<T>;
  static_assert(b128_clean([](uint32_t l) { return T::row(0, 0, l % 16) * 128 + ((l / 16) ^ T::key_a(l % 16)) * 16; }) &&
                    b128_clean([](uint32_t l) { return l % 16 * 128 + ((l / 16) ^ T::key_t(l % 16)) * 16; }),
                "fragment reads");
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t row0 = tile / tok_blocks * T::HR, tok0 = tile % tok_blocks * T::BT;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wr = wave / T::WT, wt = wave % T::WT, lr = lane & 15u, lk = lane >> 4;
  const uint32_t kcs = pk / 256, rowb = pk / 2;

  // Copies: 8 rows x 128 B each, lane l takes the piece of row l / 8 that
  // belongs at its position l % 8. Rows past the last re-read it (their
  // outputs are not stored).
  uint32_t off[T::PerWave];
#pragma unroll
  for (uint32_t u = 0; u < T::PerWave; ++u) {
    const uint32_t unit = min(wave + u * T::W, T::Units - 1), R = unit * 8 + (lane >> 3), p = lane & 7u;
    if (unit < T::BR / 8)
      off[u] = min(row0 + R % T::HR, rows - 1) * rowb + (p ^ T::key_w(R)) * 16;
    else
      off[u] = min(tok0 + R - T::BR, m - 1) * rowb + (p ^ T::key_t(R - T::BR)) * 16;
  }
  // scale copies: unit v is half (v % 2) of stripe v / 2, gate / up / token stripes in turn
  const uint32_t wstripes = (n + 127) / 128, xstripes = (m + 127) / 128, stripe = 128 * (pk / 16);
  uint32_t soff[S::PerWave];
#pragma unroll
  for (uint32_t u = 0; u < S::PerWave; ++u) {
    const uint32_t v = min(wave + u * T::W, S::Units - 1), st = v / 2;
    const uint32_t i = st < S::A ? min(row0 / 128 + st % S::PerPart, wstripes - 1)
                                 : min(tok0 / 128 + (st - S::A), xstripes - 1);
    soff[u] = i * stripe + (v % 2) * 1024 + lane * 16;
  }
  auto issue = [&](uint32_t kc_in, uint8_t* slot) __attribute__((always_inline)) {
    const uint32_t kc = min(kc_in, kcs - 1);
#pragma unroll
    for (uint32_t u = 0; u < T::PerWave; ++u) {
      const uint32_t unit = min(wave + u * T::W, T::Units - 1);  // wave-uniform
      const uint8_t* base = pick(unit >= T::BR / 8, xc, pick(T::Paired && unit >= T::HR / 8, uc, wc));
      copy16<Dma>(base + size_t(kc) * 128 + off[u], slot + unit * 1024);
    }
#pragma unroll
    for (uint32_t u = 0; u < S::PerWave; ++u) {
      const uint32_t v = min(wave + u * T::W, S::Units - 1);
      const uint8_t* base = pick(v / 2 >= S::A, xs, pick(T::Paired && v / 2 >= S::PerPart, us, ws));
      copy16<Dma>(base + size_t(kc) * 2048 + soff[u], slot + T::RowBytes + v * 1024);
    }
  };

  f4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f4{0, 0, 0, 0};
  // scale bytes of the lane's rows and tokens for element blocks 2 lk, 2 lk + 1
  // (piece lk); piece 4 + lk is 1024 B further
  uint32_t sa[NI], sb[NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const uint32_t R = T::row(wr, i, lr), rr = R % T::HR;
    sa[i] = T::RowBytes + (R / T::HR * S::PerPart + rr / 128) * 2048 + S::byte((row0 + rr) % 128, 2 * lk);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint32_t t = wt * 16 * NJ + j * 16 + lr;
    sb[j] = T::RowBytes + (S::A + t / 128) * 2048 + S::byte((tok0 + t) % 128, 2 * lk);
  }

  auto compute = [&](const uint8_t* slot) __attribute__((always_inline)) {
    const uint8_t* xl = slot + T::BR * 128;
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
      u4 ra[NI], rb[NJ];
      h2 ca[NI], cb[NJ];
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        ra[i] = *reinterpret_cast<const u4*>(slot + T::row(wr, i, lr) * 128 + (((h * 4 + lk) ^ T::key_a(lr)) * 16));
        ca[i] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(*reinterpret_cast<const uint16_t*>(slot + sa[i] + h * 1024), 1.f, false);
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        rb[j] = *reinterpret_cast<const u4*>(xl + (wt * 16 * NJ + j * 16 + lr) * 128 + (((h * 4 + lk) ^ T::key_t(lr)) * 16));
        cb[j] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(*reinterpret_cast<const uint16_t*>(slot + sb[j] + h * 1024), 1.f, false);
      }
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        half8 af[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) af[i] = widen4(ra[i][d], ca[i][d / 2]);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const half8 bf = widen4(rb[j][d], cb[j][d / 2]);
#pragma unroll
          for (int i = 0; i < NI; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf, acc[i][j], 0, 0, 0);
        }
      }
    }
  };

  // Ring: chunk kc is awaited (NS - 2 younger chunks may stay in flight), the
  // barrier publishes it and retires chunk kc - 1, whose slot takes chunk
  // kc + NS - 1. Copies past the end re-read the last chunk into a retired slot.
  constexpr int Copies = T::PerWave + S::PerWave;
  auto run = [&](uint8_t* s0, uint8_t* s1, uint8_t* s2, uint8_t* s3, uint8_t*) __attribute__((always_inline)) {
    uint8_t* const sl[4] = {s0, s1, s2, s3};
    ring<NS>(
        kcs, [&](uint32_t kc, auto ic) __attribute__((always_inline)) { issue(kc, sl[ic]); },
        [&](uint32_t kc, auto ic) __attribute__((always_inline)) {
          copies_barrier<(NS - 2) * Copies>();
          issue(kc + NS - 1, sl[(ic + NS - 1) % NS]);
          compute(sl[ic]);
        });
  };
  with_slots(lds, lds + S::Slot, lds + (NS > 2 ? 2 : 0) * S::Slot, lds + (NS > 3 ? 3 : 0) * S::Slot, lds, run);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy outlives the block

  // Lane: rows r .. r + 4 H - 1 of token lr of each token tile.
  const float factor = load_f32<Dma>(fo), factor_u = T::Paired ? load_f32<Dma>(fu) : 0.f;
  const uint32_t r = row0 + wr * (16 * H) + lk * (4 * H);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint32_t t = tok0 + wt * 16 * NJ + j * 16 + lr;
    if (t >= m) continue;
#pragma unroll
    for (int i = 0; i < H; ++i) {
      if (r + 4 * i >= n) continue;  // n % 8 == 0: whole 4-row groups
      const size_t o = size_t(t) * n + r + 4 * i;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = factor * acc[i][j][e];
      if constexpr (T::Paired) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = silu(v[e]) * (factor_u * acc[i + H][j][e]);
        store_bf16_run<4>(static_cast<uint16_t*>(y) + o, v, vec);
        continue;
      }
      if (epi == QW38_DECODE_STORE_BF16) {
        store_bf16_run<4>(static_cast<uint16_t*>(y) + o, v, vec);
        continue;
      }
      if (epi == QW38_DECODE_RESIDUAL_ADD_FP32) {
        const float4 q = *reinterpret_cast<const float4*>(residual + o);
        v[0] = q.x + v[0];
        v[1] = q.y + v[1];
        v[2] = q.z + v[2];
        v[3] = q.w + v[3];
      }
      *reinterpret_cast<float4*>(static_cast<float*>(y) + o) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

}  // namespace

hipError_t launch_pack_nvfp4(const uint16_t* x, uint32_t m, uint32_t k, uint8_t* codes,
                             uint8_t* scales, hipStream_t s) {
  const uint32_t pk = (k + 255) / 256 * 256;
  const dim3 grid(uint32_t(uint64_t((m + 127) / 128 * 128) * (pk / 8) / 256));
  if (aligned16(x) && k % 8 == 0)
    hipLaunchKernelGGL(pack_nvfp4_kernel<true>, grid, dim3(256), 0, s, x, m, k, pk, codes, scales);
  else
    hipLaunchKernelGGL(pack_nvfp4_kernel<false>, grid, dim3(256), 0, s, x, m, k, pk, codes, scales);
  return hipGetLastError();
}

hipError_t launch_nvfp4_gemv(const uint8_t* ca, const uint8_t* sa, const uint8_t* cb,
                             const uint8_t* sb, uint32_t n, uint32_t pn, uint32_t k, uint32_t pk,
                             const uint16_t* x, void* ya, void* yb, const float* ra, const float* rb,
                             int epilogue, hipStream_t s) {
  const dim3 grid((pn + 127) / 128 * 8);
  const size_t lds = size_t(pk) * 2;
  if (cb)
    hipLaunchKernelGGL(nvfp4_gemv_kernel<true>, grid, dim3(256), lds, s, ca, sa, cb, sb, n,
                       pn, k, pk, x, ya, yb, ra, rb, epilogue);
  else
    hipLaunchKernelGGL(nvfp4_gemv_kernel<false>, grid, dim3(256), lds, s, ca, sa, cb, sb,
                       n, pn, k, pk, x, ya, yb, ra, rb, epilogue);
  return hipGetLastError();
}

namespace {
struct GemmArgs {
  const uint8_t *wc, *ws, *uc, *us, *fo, *fu;
  uint32_t n, rows, pk;
  const uint8_t *xc, *xs;
  uint32_t m;
  void* y;
  const float* residual;
  int epi;
  bool dma, vec;
  hipStream_t s;
};

template <class T, bool Dma>
hipError_t gemm_tile(const GemmArgs& a) {
  constexpr int lds = T::NS * int(Scales<T>::Slot);
  const hipError_t e = set_max_lds(reinterpret_cast<const void*>(&nvfp4_gemm_kernel<T, Dma>), lds);
  if (e != hipSuccess) return e;
  const uint32_t tb = (a.m + T::BT - 1) / T::BT;
  hipLaunchKernelGGL((nvfp4_gemm_kernel<T, Dma>), dim3((a.n + T::HR - 1) / T::HR * tb), dim3(T::W * 64), lds, a.s,
                     a.wc, a.ws, a.uc, a.us, a.fo, a.fu, a.n, a.rows, a.pk, a.xc, a.xs, a.m, a.y, a.residual, a.epi,
                     a.vec, tb);
  return hipGetLastError();
}

// Tile by the busiest CU's time per 256 elements of K, in microseconds with
// one, two and three blocks on it, measured at K = 5120. Over 110 sizes
// (n 1024..17408, 2..1024 tokens) the choice takes at most 2% longer than the
// best tile plain and 7% paired, 0.3% and 2% on average. The 128-row tiles with two
// blocks on a CU serve the large grids (paired 17408 features x 1024 tokens
// 1304 -> 411 us with the activation pack, 890 TFLOP/s); smaller tiles fill the CUs
// for fewer rows or tokens, and the 16-token ones keep three chunks in flight
// for the weight stream (paired 17408 features at 16 tokens: 331 -> 42 us).
constexpr TileCost kNvfp4Cost[] = {{128, 128, 2, {2.4f, 4.35f}}, {128, 64, 2, {1.45f, 2.55f}},
                                   {64, 64, 3, {0.97f, 1.6f, 2.27f}}, {128, 32, 2, {1.0f, 1.55f}},
                                   {64, 32, 2, {0.74f, 1.1f}},   {128, 16, 1, {0.76f}},
                                   {64, 16, 2, {0.67f, 1.05f}}};

template <bool P>
hipError_t gemm(const GemmArgs& a) {
  // Spans that are not 16-byte aligned (qw38_prefill_mlp takes any) are staged
  // through registers.
  if (!a.dma) return gemm_tile<Tile<2, 2, 2, 2, 2, P>, false>(a);
#define QW38_NV(...) return gemm_tile<Tile<__VA_ARGS__, P>, true>(a)
  switch (nvfp4_gemm_plan(P, a.n, a.m, uint32_t(cu_count())).tile) {
    case 0: QW38_NV(2, 4, 4, 2, 2);
    case 1: QW38_NV(2, 2, 4, 2, 2);
    case 2: QW38_NV(2, 2, 2, 2, 2);
    case 3: QW38_NV(4, 1, 2, 2, 3);
    case 4: QW38_NV(2, 2, 2, 1, 4);
    case 5: QW38_NV(4, 1, 2, 1, 4);
    default: QW38_NV(2, 1, 2, 1, 4);
  }
#undef QW38_NV
}
}  // namespace

GemmPlan nvfp4_gemm_plan(bool paired, uint32_t n, uint32_t m, uint32_t cus) {
  return {0, pick_tile(kNvfp4Cost, uint64_t(n) * (paired ? 2 : 1), m, cus).index, uint32_t(std::size(kNvfp4Cost))};
}

hipError_t launch_nvfp4_gemm(const uint8_t* wc, const uint8_t* wsf, const float* wfactor,
                             uint32_t n, uint32_t code_rows, uint32_t pk, const uint8_t* xc,
                             const uint8_t* xs, uint32_t m, void* y, const float* residual,
                             int epilogue, hipStream_t s) {
  GemmArgs a{};
  a.wc = wc, a.ws = wsf, a.fo = reinterpret_cast<const uint8_t*>(wfactor);
  a.n = n, a.rows = code_rows, a.pk = pk, a.xc = xc, a.xs = xs, a.m = m;
  a.y = y, a.residual = residual, a.epi = epilogue;
  a.dma = aligned16(wc) && aligned16(wsf) && aligned16(xc) && aligned16(xs);
  a.vec = aligned16(y) || (epilogue == QW38_DECODE_STORE_BF16 && reinterpret_cast<uintptr_t>(y) % 8 == 0);
  a.s = s;
  return gemm<false>(a);
}

hipError_t launch_nvfp4_paired(const uint8_t* gc, const uint8_t* gsf, const uint8_t* uc, const uint8_t* usf,
                               uint32_t n, uint32_t code_rows, uint32_t pk, const uint8_t* xc,
                               const uint8_t* xs, uint32_t m, uint16_t* y, hipStream_t s) {
  GemmArgs a{};
  a.wc = gc, a.ws = gsf + 256, a.fo = gsf, a.uc = uc, a.us = usf + 256, a.fu = usf;
  a.n = n, a.rows = code_rows, a.pk = pk, a.xc = xc, a.xs = xs, a.m = m, a.y = y;
  a.dma = aligned16(gc) && aligned16(gsf) && aligned16(uc) && aligned16(usf) && aligned16(xc) && aligned16(xs);
  a.vec = reinterpret_cast<uintptr_t>(y) % 8 == 0;
  a.s = s;
  return gemm<true>(a);
}

}  // namespace qw38hip
