// Exact dequantization of pool rows to bf16, shared by the sparse attention and the gathers.
#pragma once

#include "kvt_common.h"

namespace kvt {

// bf16 pair (round to nearest even, one v_cvt_pk_bf16_f32): lo in bits 0-15.
KVT_DEV uint32_t bf16x2(float lo, float hi) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v){lo, hi}, bf2v));
}

// Eight channels of one row, dequantized: bf16((c * s) * sm) for code c, the row's fp16 scale s (bits sbits) and the
// channel's smoothing factor sm, as the gathers write them.  INT8 rows give 8 bytes of codes, INT4 rows 4 (byte j =
// channel 2 j in the low nibble, 2 j + 1 in the high one, stored as c + 8).  A code with offset o (c + o >= 0) goes
// into the mantissa of an fp16 magic value h = 1024 + (c + o) (v_perm_b32 for bytes, v_and_or_b32 for nibbles), in
// pairs of channels (0, 2), (1, 3), (4, 6), (5, 7); v_fma_mix_f32 converts h and s and computes
// h * s - (1024 + o) * s in one rounding, whose exact value c * s is representable (4 or 8 bits times the scale's
// 11), so the fp32 product equals the plain c * s; the caller then multiplies by the smoothing factor in fp32 and
// rounds each pair to nearest even with v_cvt_pk_bf16_f32.
KVT_DEV uint32_t and_or(uint32_t x, uint32_t m, uint32_t o) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "s"(m), "v"(o));
  return r;
}
KVT_DEV float mix(uint32_t w, int half, _Float16 s, float c) {
  typedef _Float16 h2v __attribute__((ext_vector_type(2)));
  return fmaf((float)__builtin_bit_cast(h2v, w)[half], (float)s, c);
}
KVT_DEV void magic8(uint2 w, uint32_t m[4]) {
  const uint32_t u = w.x ^ 0x80808080u, v = w.y ^ 0x80808080u;
  m[0] = __builtin_amdgcn_perm(0x64646464u, u, 0x04020400u);
  m[1] = __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u);
  m[2] = __builtin_amdgcn_perm(0x64646464u, v, 0x04020400u);
  m[3] = __builtin_amdgcn_perm(0x64646464u, v, 0x04030401u);
}
KVT_DEV void magic4(uint32_t w, uint32_t m[4]) {   // pairs (0, 4), (1, 5), (2, 6), (3, 7), one instruction less than magic8's
  m[0] = and_or(w, 0x000F000Fu, 0x64006400u);
  m[1] = and_or(w >> 4, 0x000F000Fu, 0x64006400u);
  m[2] = and_or(w >> 8, 0x000F000Fu, 0x64006400u);
  m[3] = and_or(w >> 12, 0x000F000Fu, 0x64006400u);
}

}  // namespace kvt
