// FP8 (OCP E4M3FN) path of qw38's prefill and decode (cuda/fp8.hpp, cuda/fp8.cu):
//   pack_fp8    BF16 [m][k] -> E4M3 codes [pm][pk] + FP32 scales [pk/128][pm],
//               one scale per (row, 128-column block) = absmax / 448
//               (cuda/fp8.cu:64-81);
//   fp8 GEMV    y[r] = sum_c value(w[r][c]) * s[c/128][r/128] * x[c], BF16 x,
//               the decode_mmv layout 0x020F (cuda/fp8.cu:82-112, 184-203);
//   fp8 GEMM    y[t][r] = sum over 128-column blocks of sx[b][t] * sw[b][r/128]
//               * sum_c value(x[t][c]) value(w[r][c]) (cuda/fp8.cu:137-160).
//
// The GEMM runs on FP16 MFMAs, not the FP8 ones: on gfx950 the FP8 matrix
// instructions (16x16x32 fp8, 16x16x128 f8f6f4) align the products of a dot
// into a narrow accumulator and lose about 1e-4 of the sum of |products| on
// realistic packed data, while every E4M3 value is exact in FP16 and the FP16
// MFMA keeps the sum to about 1e-7 (the reference's budget is 1e-5 of it,
// tests/fp8_test.cpp:100). Codes are staged in LDS as bytes and widened to
// FP16 per fragment with v_cvt_scalef32_pk_f16_fp8 (scale 1: exact; it issues
// at the rate of an FMA, two codes each).
#include "lds_gemm.hpp"

namespace qw38hip {
namespace {

// Maximum over groups of N = 16 or 64 lanes, all active: within a row of 16 by
// DPP moves (a shuffle goes through LDS and takes several times as long).
template <int N>
__device__ __forceinline__ float lanes_max(float v) {
  auto step = [&](auto ctrl) __attribute__((always_inline)) {
    const int x = __float_as_int(v);
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, decltype(ctrl)::value, 0xf, 0xf, true)));
  };
  step(std::integral_constant<int, 0xb1>{});   // quad_perm 1 0 3 2
  step(std::integral_constant<int, 0x4e>{});   // quad_perm 2 3 0 1
  step(std::integral_constant<int, 0x141>{});  // row_half_mirror
  step(std::integral_constant<int, 0x140>{});  // row_mirror
  if constexpr (N == 64) {
    v = fmaxf(v, __shfl_xor(v, 16));
    v = fmaxf(v, __shfl_xor(v, 32));
  }
  return v;
}

// ---- pack: E elements per thread, 128 / E threads per 128-column block. With
// eight, 16-byte loads and four cross-lane steps: 512 x 5120 10.5 -> 6.9 us (one
// element per thread before). With two, a thread's chain of divides is short, which
// is the time of few rows.
template <bool Vec, int E>
__global__ __launch_bounds__(256) void pack_fp8_kernel(const uint16_t* __restrict__ x, uint32_t m,
                                                       uint32_t k, uint32_t pm, uint32_t pk,
                                                       uint8_t* __restrict__ codes,
                                                       float* __restrict__ scales) {
  uint32_t r, c;
  if constexpr (E == 2) {  // grid (pm / 4, pk / 128), a wave per block of 128: no division in the short kernel
    r = blockIdx.x * 4 + (threadIdx.x >> 6);
    c = blockIdx.y * 128 + (threadIdx.x & 63u) * 2;
  } else {  // the grid is pm whole rows
    const uint32_t per_row = pk / E, t = blockIdx.x * 256 + threadIdx.x;
    r = t / per_row;
    c = t % per_row * E;
  }
  float v[E];
  const uint16_t* row = x + size_t(r < m ? r : 0) * k;
  if constexpr (E == 8) {
    load8_bf16<Vec>(row, c, k, r < m, v);
  } else {
#pragma unroll
    for (int i = 0; i < E; ++i) v[i] = r < m && c + i < k ? bf16_to_f32(row[c + i]) : 0.f;
  }
  float peak = 0.f;
#pragma unroll
  for (int i = 0; i < E; ++i) peak = fmaxf(peak, isfinite(v[i]) ? fabsf(v[i]) : __builtin_inff());
  peak = lanes_max<128 / E>(peak);
  // nonfinite blocks carry NaN (cuda/fp8.cu:75-77)
  const float scale = isfinite(peak) ? (peak == 0.f ? 1.f : fmaxf(__fdiv_rn(peak, 448.f), 0x1p-126f))
                                     : __builtin_nanf("");
  if (threadIdx.x % (128 / E) == 0) scales[size_t(c / 128) * pm + r] = scale;
  uint32_t w[2] = {0u, 0u};
#pragma unroll
  for (int i = 0; i < E; ++i) w[i / 4] |= e4m3_rne(__fdiv_rn(v[i], scale)) << (8 * (i % 4));
  if constexpr (E == 8) *reinterpret_cast<uint2*>(codes + size_t(r) * pk + c) = make_uint2(w[0], w[1]);
  else *reinterpret_cast<uint16_t*>(codes + size_t(r) * pk + c) = uint16_t(w[0]);
}

// ---- decode GEMV: one wave per row, 16 contiguous codes per lane ----
__device__ __forceinline__ float dot16(const uint4 c, const uint32_t* xw) {
  // codes 16 E4M3 (c), x 16 BF16 as 8 pairs (xw)
  const uint32_t cw[4] = {c.x, c.y, c.z, c.w};
  float p = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float w[4] = {__builtin_amdgcn_cvt_f32_fp8(int(cw[i]), 0), __builtin_amdgcn_cvt_f32_fp8(int(cw[i]), 1),
                        __builtin_amdgcn_cvt_f32_fp8(int(cw[i]), 2), __builtin_amdgcn_cvt_f32_fp8(int(cw[i]), 3)};
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const uint32_t pair = xw[2 * i + (b >> 1)];
      const float xv = __uint_as_float((b & 1) ? (pair & 0xffff0000u) : (pair << 16));
      p = fmaf(w[b], xv, p);
    }
  }
  return p;
}

__device__ __forceinline__ void gemv_store(float acc, uint32_t row, void* y, const float* residual, int epi) {
  if (epi == QW38_DECODE_STORE_BF16) {
    static_cast<uint16_t*>(y)[row] = f32_to_bf16_rne(acc);
  } else if (epi == QW38_DECODE_RESIDUAL_ADD_FP32) {
    float* dst = y ? static_cast<float*>(y) : const_cast<float*>(residual);
    dst[row] = acc + residual[row];
  } else {
    static_cast<float*>(y)[row] = acc;
  }
}

// K <= 1024 C: a wave takes Rows consecutive rows, 16 contiguous codes per
// lane and 1 KB chunk, all loaded before the first is summed. The lane's inputs
// go straight to registers and serve all its rows, so the weight stream never
// waits for a staging barrier. Products of an E4M3 value (exact in BF16) and a
// BF16 input meet in v_dot2_f32_bf16.
// Bound: HBM. With and without this kernel (x staged in LDS, two chunks in
// flight), weights not cached: 12288 x 5120 14.1 and 22.1 us (4.5 TB/s), 1024 x 5120
// 3.1 and 5.6, 17408 x 1024 6.3 and 10.0, 5120 x 6144 8.7 and 9.4.
typedef __bf16 bfx2 __attribute__((ext_vector_type(2)));
template <int C, bool Vec, uint32_t Rows>
__global__ __launch_bounds__(256) void fp8_gemv_rows_kernel(const uint8_t* __restrict__ codes,
                                                            const float* __restrict__ scales, uint32_t n,
                                                            uint32_t k, const uint16_t* __restrict__ x,
                                                            void* y, const float* residual, int epi) {
  const uint32_t lane = threadIdx.x & 63u, nb = n / 128;
  const uint32_t r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * Rows;  // Rows divides n
  if (r0 >= n) return;
  u4 w[Rows][C];
  auto load = [&](uint32_t row, int o) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint32_t col = c * 1024 + lane * 16;
      const u4 v = *reinterpret_cast<const u4*>(codes + size_t(row) * k + (col < k ? col : 0u));
      w[o][c] = col < k ? v : u4{0u, 0u, 0u, 0u};
    }
  };
  // Rows divides 128: one row block of scales per wave
  float sc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const uint32_t b = c * 8 + (lane >> 3);
    sc[c] = scales[size_t(b * 128 < k ? b : 0u) * nb + r0 / 128];
  }
  load(r0, 0);
  u4 xv[C][2];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const uint32_t col = c * 1024 + lane * 16;
    if constexpr (Vec) {
#pragma unroll
      for (int h = 0; h < 2; ++h) xv[c][h] = *reinterpret_cast<const u4*>(x + (col < k ? col + 8 * h : 0u));
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        xv[c][i / 4][i % 4] = col < k ? uint32_t(x[col + 2 * i]) | uint32_t(x[col + 2 * i + 1]) << 16 : 0u;
    }
  }
  auto row_sum = [&](uint32_t row, int o) __attribute__((always_inline)) {
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int c = 0; c < C; ++c) {
      float p = 0.f, q = 0.f;  // two chains: half the roundings each
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bfx2 lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(int(w[o][c][i]), 1.f, false);
        const bfx2 hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(int(w[o][c][i]), 1.f, true);
        p = __builtin_amdgcn_fdot2_f32_bf16(lo, __builtin_bit_cast(bfx2, uint32_t(xv[c][i / 2][i % 2 * 2])), p, false);
        q = __builtin_amdgcn_fdot2_f32_bf16(hi, __builtin_bit_cast(bfx2, uint32_t(xv[c][i / 2][i % 2 * 2 + 1])), q, false);
      }
      // lanes past K hold zeros and another block's scale
      part[c % 2] = c * 1024 + lane * 16 < k ? fmaf(sc[c], p + q, part[c % 2]) : part[c % 2];
    }
    float acc = part[0] + part[1];
    // the last steps in FP64, where a rounding costs most: the relative error
    // at 12288 x 5120 stays below that of 16-step FP32 chains (8.12e-8)
#pragma unroll
    for (int o2 = 32; o2 > 4; o2 >>= 1) acc += __shfl_xor(acc, o2);
    double sum = acc;
#pragma unroll
    for (int o2 = 4; o2 > 0; o2 >>= 1) sum += __shfl_xor(sum, o2);
    if (lane == 0) gemv_store(float(sum), row, y, residual, epi);
  };
  if constexpr (Rows == 2) load(r0 + 1, 1);
#pragma unroll
  for (uint32_t i = 0; i < Rows; ++i) row_sum(r0 + i, i);
}

// Any K: one wave per row, the input in LDS, two chunks in flight.
__global__ __launch_bounds__(256) void fp8_gemv_kernel(const uint8_t* __restrict__ codes,
                                                       const float* __restrict__ scales, uint32_t n,
                                                       uint32_t k, const uint16_t* __restrict__ x,
                                                       void* y, const float* residual, int epi) {
  extern __shared__ __align__(16) uint8_t smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
  for (uint32_t i = threadIdx.x; i < k; i += 256) xs[i] = x[i];
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= n) return;
  const uint8_t* rp = codes + size_t(row) * k;
  const float* sp = scales + row / 128;
  const uint32_t nb = n / 128;
  float acc = 0.f;
  uint32_t base = lane * 16;
  // two 1 KB rows spans per iteration in flight
  for (; base + 1024 < k; base += 2048) {
    const uint4 c0 = *reinterpret_cast<const uint4*>(rp + base);
    const uint4 c1 = *reinterpret_cast<const uint4*>(rp + base + 1024);
    const float s0 = sp[size_t(base / 128) * nb], s1 = sp[size_t((base + 1024) / 128) * nb];
    const uint4* x0 = reinterpret_cast<const uint4*>(xs + base);
    const uint4* x1 = reinterpret_cast<const uint4*>(xs + base + 1024);
    const uint4 a0 = x0[0], a1 = x0[1], b0 = x1[0], b1 = x1[1];
    const uint32_t xa[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    const uint32_t xb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
    acc = fmaf(s0, dot16(c0, xa), acc);
    acc = fmaf(s1, dot16(c1, xb), acc);
  }
  if (base < k) {
    const uint4 c0 = *reinterpret_cast<const uint4*>(rp + base);
    const uint4* x0 = reinterpret_cast<const uint4*>(xs + base);
    const uint4 a0 = x0[0], a1 = x0[1];
    const uint32_t xa[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    acc = fmaf(sp[size_t(base / 128) * nb], dot16(c0, xa), acc);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if (lane == 0) gemv_store(acc, row, y, residual, epi);
}

// ---- GEMM ----
// Widens two dwords (eight codes) to one FP16 fragment, exactly.
__device__ __forceinline__ half8 widen(uint32_t x, uint32_t y) {
  const h2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(x), 1.f, false);
  const h2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(x), 1.f, true);
  const h2 c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(y), 1.f, false);
  const h2 d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(int(y), 1.f, true);
  return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}

// One ring slot holds a 128-column block: the raw codes (lds_gemm.hpp), then
// the tile's BT token scales of that block. P sums a block on the matrix cores and
// one FMA per output scales it: acc = fma(sw * sx[token], P, acc). Every tile
// runs the same chain per output, so its shape never changes a bit.
//
// Bound: the matrix cores (16 cycles per MFMA; 36% busy) beside 4 VALU
// instructions per MFMA for widening and scaling, which mostly run beside and
// not under them. No LDS bank conflicts. Copies take no registers and
// no VALU work, one barrier covers a whole 128-column block, and the 128-row
// tiles keep two blocks of eight waves on a CU. 12288 x 5120, weights not cached:
// 236 -> 72 us at 512 tokens (273 -> 900 TFLOP/s), 377 -> 128 at 1024, 137 -> 17 at 16
// (3.7 TB/s).
template <class T>
__global__ __launch_bounds__(T::W * 64) void fp8_gemm_kernel(
    const uint8_t* __restrict__ wc, const float* __restrict__ ws, uint32_t n, uint32_t k,
    const uint8_t* __restrict__ xc, const float* __restrict__ xsc, uint32_t m, void* __restrict__ y,
    const float* __restrict__ residual, uint32_t valid, int epi, uint32_t tok_blocks) {
  constexpr int NI = T::NI, NJ = T::NJ, NS = T::NS;
  constexpr uint32_t Slot = T::RowBytes + 1024;
  static_assert(b128_clean([](uint32_t l) { return T::row(0, 0, l % 16) * 128 + ((l / 16) ^ T::key_a(l % 16)) * 16; }) &&
                    b128_clean([](uint32_t l) { return l % 16 * 128 + ((l / 16) ^ T::key_t(l % 16)) * 16; }),
                "fragment reads");
  extern __shared__ __align__(16) uint8_t lds[];
  const uint32_t tile = xcd_tile(blockIdx.x, gridDim.x);
  const uint32_t row0 = tile / tok_blocks * T::BR, tok0 = tile % tok_blocks * T::BT;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wr = wave / T::WT, wt = wave % T::WT, lr = lane & 15u, lk = lane >> 4;
  const uint32_t kbs = k / 128;

  // Copies: 8 rows x 128 B each, lane l takes the piece of row l / 8 that
  // belongs at its position l % 8. Rows past n re-read the last one.
  uint32_t off[T::PerWave];
#pragma unroll
  for (uint32_t u = 0; u < T::PerWave; ++u) {
    const uint32_t unit = min(wave + u * T::W, T::Units - 1), R = unit * 8 + (lane >> 3), p = lane & 7u;
    if (unit < T::BR / 8)
      off[u] = min(row0 + R, n - 1) * k + (p ^ T::key_w(R)) * 16;
    else
      off[u] = (tok0 + R - T::BR) * k + (p ^ T::key_t(R - T::BR)) * 16;
  }
  auto issue = [&](uint32_t kb_in, uint8_t* slot) __attribute__((always_inline)) {
    const uint32_t kb = min(kb_in, kbs - 1);
#pragma unroll
    for (uint32_t u = 0; u < T::PerWave; ++u) {
      const uint32_t unit = min(wave + u * T::W, T::Units - 1);  // wave-uniform
      copy16<true>(pick(unit < T::BR / 8, wc, xc) + size_t(kb) * 128 + off[u], slot + unit * 1024);
    }
    // token scales: every wave copies the same 1 KB, BT floats and repeats of the last four
    copy16<true>(reinterpret_cast<const uint8_t*>(xsc + size_t(kb) * m + tok0 + min(lane, T::BT / 4 - 1) * 4),
                 slot + T::RowBytes);
  };

  f4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f4{0, 0, 0, 0};
  // Weight scales of the tile's row blocks, all of K, once: a load in the loop
  // would queue behind the copies in flight. A lane's rows 4 lk NI .. +4 NI - 1
  // lie in row blocks b0 and b1 (of at most three).
  const uint32_t nbs = n / 128, rb0 = row0 / 128;
  float* swt = reinterpret_cast<float*>(lds + NS * Slot);  // [kbs][4]
  for (uint32_t i = threadIdx.x; i < kbs * 4; i += T::W * 64)
    swt[i] = ws[size_t(i / 4) * nbs + min(rb0 + i % 4, nbs - 1)];
  const uint32_t lrow = row0 + wr * 16 * NI + lk * 4 * NI;
  const uint32_t b0 = lrow / 128 - rb0, b1 = (lrow + 4 * NI - 4) / 128 - rb0;

  auto compute = [&](uint32_t kb, const uint8_t* slot, const float* swt) __attribute__((always_inline)) {
    f4 P[NI][NJ];
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) P[i][j] = f4{0, 0, 0, 0};
    const uint8_t* wl = slot;
    const uint8_t* xl = slot + T::BR * 128;
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
      u4 ra[NI], rb[NJ];
#pragma unroll
      for (int i = 0; i < NI; ++i)
        ra[i] = *reinterpret_cast<const u4*>(wl + T::row(wr, i, lr) * 128 + (((h * 4 + lk) ^ T::key_a(lr)) * 16));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        rb[j] = *reinterpret_cast<const u4*>(xl + (wt * 16 * NJ + j * 16 + lr) * 128 +
                                                (((h * 4 + lk) ^ T::key_t(lr)) * 16));
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        half8 af[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) af[i] = d ? widen(ra[i].z, ra[i].w) : widen(ra[i].x, ra[i].y);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const half8 bf = d ? widen(rb[j].z, rb[j].w) : widen(rb[j].x, rb[j].y);
#pragma unroll
          for (int i = 0; i < NI; ++i) P[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i], bf, P[i][j], 0, 0, 0);
        }
      }
    }
    const float sw0 = swt[kb * 4 + b0], sw1 = swt[kb * 4 + b1];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float sx = *reinterpret_cast<const float*>(slot + T::RowBytes + (wt * 16 * NJ + j * 16 + lr) * 4);
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        // only a run of 12 rows (NI = 3) can cross a row block
        const float s = (NI == 3 && (lrow + 4 * i) / 128 - rb0 != b0 ? sw1 : sw0) * sx;
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(s, P[i][j][v], acc[i][j][v]);
      }
    }
  };

  // Ring: chunk kb is awaited (NS - 2 younger chunks may stay in flight), the
  // barrier publishes it and retires chunk kb - 1, whose slot takes chunk
  // kb + NS - 1. Copies past the end re-read the last chunk into a retired slot.
  constexpr int Copies = T::PerWave + 1;
  auto run = [&](uint8_t* s0, uint8_t* s1, uint8_t* s2, uint8_t* s3, uint8_t* table) __attribute__((always_inline)) {
    uint8_t* const sl[4] = {s0, s1, s2, s3};
    ring<NS>(
        kbs, [&](uint32_t kb, auto ic) __attribute__((always_inline)) { issue(kb, sl[ic]); },
        [&](uint32_t kb, auto ic) __attribute__((always_inline)) {
          copies_barrier<(NS - 2) * Copies>();
          issue(kb + NS - 1, sl[(ic + NS - 1) % NS]);
          compute(kb, sl[ic], reinterpret_cast<const float*>(table));
        });
  };
  with_slots(lds, lds + Slot, lds + (NS > 2 ? 2 : 0) * Slot, lds + (NS > 3 ? 3 : 0) * Slot, lds + NS * Slot, run);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no copy outlives the block

  // Lane: rows r .. r + 4 NI - 1 of token lr of each token tile. epi 0 writes
  // the raw FP32 product of every padded token (fp8_gemm); the prefill
  // epilogues (cuda/prefill.cu:116-134) write only the first `valid` tokens:
  // BF16 RNE, FP32, or FP32 residual[t][r] + product.
  const uint32_t r = lrow;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint32_t t = tok0 + wt * 16 * NJ + j * 16 + lr;
    if (epi != 0 && t >= valid) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if (r + 4 * i >= n) continue;  // n % 128 == 0: whole 4-row groups
      const size_t o = size_t(t) * n + r + 4 * i;
      float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
      if (epi == QW38_DECODE_STORE_BF16) {
        store_bf16_run<4>(static_cast<uint16_t*>(y) + o, v, true);
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

__global__ void fp8_store_bf16_kernel(const float* __restrict__ x, uint16_t* __restrict__ y,
                                      uint64_t count) {
  const uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  if (i < count) y[i] = f32_to_bf16_rne(x[i]);
}

}  // namespace

hipError_t launch_pack_fp8(const uint16_t* x, uint32_t m, uint32_t k, uint8_t* codes, float* scales,
                           hipStream_t s) {
  const uint32_t pm = (m + 127) / 128 * 128, pk = (k + 127) / 128 * 128;
  // Two elements per thread up to 4608 per CU: 128 x 1024 2.6 us against 3.7 with
  // eight, 512 x 1024 3.1 and 3.8, 1024 x 1024 4.07 and 4.12; beyond, 768 x 2048
  // 4.9 and 4.6, 512 x 5120 7.0 and 5.8. pm and pk are multiples of 128.
  const bool few = uint64_t(pm) * pk <= uint64_t(cu_count()) * 4608;
  const dim3 grid = few ? dim3(pm / 4, pk / 128) : dim3(uint32_t(uint64_t(pm) * (pk / 8) / 256));
#define QW38_PACK(V, E) \
  hipLaunchKernelGGL((pack_fp8_kernel<V, E>), grid, dim3(256), 0, s, x, m, k, pm, pk, codes, scales)
  if (few) QW38_PACK(false, 2);
  else if (aligned16(x) && k % 8 == 0) QW38_PACK(true, 8);
  else QW38_PACK(false, 8);
#undef QW38_PACK
  return hipGetLastError();
}

hipError_t launch_fp8_gemv(const uint8_t* codes, const float* scales, uint32_t n, uint32_t k,
                           const uint16_t* x, void* y, const float* residual, int epilogue,
                           hipStream_t s) {
  // One row per wave up to 32 waves per CU, two beyond. In one comparison
  // (times of its own): 17408 x 5120 20.6 us with one, 20.0 with two, 22.4 with four;
  // 12288 x 5120 15.7, 15.5, 15.6; 5120 x 6144 10.2, 10.6, 12.0; 1024 x 5120 3.8, 4.6, 6.8. Up to K = 1024 one
  // chunk serves (5120 x 256 2.54 us, 2.99 as the first of two); with two rows per
  // wave it is the slower form (17408 x 1024 5.78, 5.47).
  const uint32_t rows = n > uint32_t(cu_count()) * 32 ? 2 : 1;
#define QW38_GEMV_AS(C, V, R)                                                                             \
  hipLaunchKernelGGL((fp8_gemv_rows_kernel<C, V, R>), dim3((n / R + 3) / 4), dim3(256), 0, s, codes, scales, n, k, \
                     x, y, residual, epilogue)
#define QW38_GEMV(C)                          \
  if (rows == 2) {                            \
    if (aligned16(x)) QW38_GEMV_AS(C, true, 2); \
    else QW38_GEMV_AS(C, false, 2);           \
  } else {                                    \
    if (aligned16(x)) QW38_GEMV_AS(C, true, 1); \
    else QW38_GEMV_AS(C, false, 1);           \
  }
  if (k <= 1024 && rows == 1) {
    if (aligned16(x)) QW38_GEMV_AS(1, true, 1);
    else QW38_GEMV_AS(1, false, 1);
  } else if (k <= 2048) {
    QW38_GEMV(2);
  } else if (k <= 4096) {
    QW38_GEMV(4);
  } else if (k <= 5120) {
    QW38_GEMV(5);
  } else if (k <= 6144) {
    QW38_GEMV(6);
  } else {
    hipLaunchKernelGGL(fp8_gemv_kernel, dim3((n + 3) / 4), dim3(256), size_t(k) * 2, s, codes,
                       scales, n, k, x, y, residual, epilogue);
  }
#undef QW38_GEMV
#undef QW38_GEMV_AS
  return hipGetLastError();
}

namespace {
template <class T>
hipError_t fp8_gemm_tile(const uint8_t* wc, const float* ws, uint32_t n, uint32_t k, const uint8_t* xc,
                         const float* xs, uint32_t m, void* y, const float* residual, uint32_t valid,
                         int epilogue, hipStream_t s) {
  constexpr int ring = T::NS * int(T::RowBytes + 1024);
  const int lds = ring + int(k / 128) * 16;
  const hipError_t e = set_max_lds(reinterpret_cast<const void*>(&fp8_gemm_kernel<T>), ring + 17408 / 128 * 16);
  if (e != hipSuccess) return e;
  const uint32_t tb = (valid + T::BT - 1) / T::BT;
  hipLaunchKernelGGL(fp8_gemm_kernel<T>, dim3((n + T::BR - 1) / T::BR * tb), dim3(T::W * 64), lds, s, wc, ws, n, k,
                     xc, xs, m, y, residual, valid, epilogue, tb);
  return hipGetLastError();
}
}  // namespace

namespace {
// Tile by the busiest CU's time per 128-column block, in microseconds with
// one, two, ... blocks on it, measured at K = 5120 and 6144. Over 210 shapes
// (n 128..12288, K 1024..6144, 1..1024 tokens) the choice takes 1% longer than
// the best tile on average and at most 19% (2560 x 5120 at 200 tokens; 16% in
// another run). Large grids
// take the 128 x 128 and 96 x 128 tiles; 128 x 64 and 64 x 64 fill
// the CUs where those leave them idle; the small ones, with a ring of four
// chunks in flight, are for few tokens, where the weight stream sets the
// time (12288 x 5120: 16 tokens 15.6 us on 64 x 16, 23 us on 64 x 64; 64 tokens 32.1
// and 25.4).
constexpr TileCost kFp8Cost[] = {{128, 128, 2, {1.13f, 2.2f}},
                                 {96, 128, 2, {0.95f, 1.72f}},
                                 {128, 64, 3, {0.71f, 1.2f, 1.8f}},
                                 {64, 64, 3, {0.52f, 0.79f, 1.09f}},
                                 {64, 16, 5, {0.33f, 0.44f, 0.65f, 0.78f, 0.95f}},
                                 {32, 16, 8, {0.285f, 0.355f, 0.385f, 0.41f, 0.57f, 0.86f, 0.87f, 0.93f}}};
}  // namespace

GemmPlan fp8_gemm_plan(uint32_t n, uint32_t m, uint32_t cus) {
  return {0, pick_tile(kFp8Cost, n, m, cus).index, uint32_t(std::size(kFp8Cost))};
}

hipError_t launch_fp8_gemm(const uint8_t* wc, const float* ws, uint32_t n, uint32_t k,
                           const uint8_t* xc, const float* xs, uint32_t m, void* y,
                           const float* residual, uint32_t valid, int epilogue, hipStream_t s) {
#define QW38_FP8(...) return fp8_gemm_tile<Tile<__VA_ARGS__, false>>(wc, ws, n, k, xc, xs, m, y, residual, valid, epilogue, s)
  switch (fp8_gemm_plan(n, valid, uint32_t(cu_count())).tile) {
    case 0: QW38_FP8(4, 2, 2, 4, 2);
    case 1: QW38_FP8(2, 4, 3, 2, 2);
    case 2: QW38_FP8(4, 2, 2, 2, 2);
    case 3: QW38_FP8(2, 2, 2, 2, 3);
    case 4: QW38_FP8(4, 1, 1, 1, 4);
    default: QW38_FP8(2, 1, 1, 1, 4);
  }
#undef QW38_FP8
}

hipError_t launch_fp8_store_bf16(const float* x, uint16_t* y, uint64_t count, hipStream_t s) {
  hipLaunchKernelGGL(fp8_store_bf16_kernel, dim3(uint32_t((count + 255) / 256)), dim3(256), 0, s, x,
                     y, count);
  return hipGetLastError();
}

}  // namespace qw38hip
