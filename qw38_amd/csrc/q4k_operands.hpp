// BF16 weight operands of Q4_K (layout 0x020D), shared by the BF16 decode GEMV
// and the BF16 prefill.
#pragma once

#include "common.hpp"

namespace qw38hip {

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float fl2 __attribute__((ext_vector_type(2)));

// Eight weight operands BF16_RNE(fma(d s, c, -d_min m)) of one code word (byte
// b: codes 2b, 2b + 1). A nibble masked in place in a 16-bit half is the FP16
// subnormal c 2^-24 (or c 2^-20 four bits higher), which v_fma_mix_f32 takes
// as an operand: with ds scaled by that power (exact) the product is the
// same, and no code is converted first. 17 instructions against 23.
__device__ __forceinline__ bf8 operands8(uint32_t w, float ds24, float ds20, float ndm) {
  const uint32_t w8 = w >> 8;
  const uint32_t v[4] = {w & 0x000f000fu, w & 0x00f000f0u, w8 & 0x000f000fu, w8 & 0x00f000f0u};
  float c[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const h2 h = __builtin_bit_cast(h2, v[i]);
    const float ds = i & 1 ? ds20 : ds24;
    c[i] = fmaf(ds, float(h[0]), ndm);
    c[4 + i] = fmaf(ds, float(h[1]), ndm);
  }
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((fl2{c[2 * i], c[2 * i + 1]}), bf2));
  return __builtin_bit_cast(bf8, u4{o[0], o[1], o[2], o[3]});
}

}  // namespace qw38hip
