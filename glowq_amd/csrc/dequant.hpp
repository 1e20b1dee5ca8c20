// A code word as the B operand of the matrix instructions.
#pragma once

#include "common.hpp"

namespace glowq {

// 8 codes of one word -> fp16((code - zero) * scale), in nibble order (0,4,1,5,2,6,3,7); kScaled = false: code - zero, exact.
// zb_lo = -(1024 + zero), zb_hi = -(64 + zero), both exact in fp16.
template <bool kScaled = true>
__device__ __forceinline__ h8 dequant_word(uint32_t w, h2 zb_lo, h2 zb_hi, h2 s2) {
  // the two exponent patterns (1024.0 and 64.0 in both halves) live in vector registers: with the nibble mask as the one
  // scalar operand the mask-and-merge is then a single v_and_or_b32 instead of an AND and an OR
  uint32_t e1024, e64;
  asm("v_mov_b32 %0, 0x64006400" : "=v"(e1024));
  asm("v_mov_b32 %0, 0x54005400" : "=v"(e64));
  const uint32_t hi = w >> 8;
  const h2 q0 = bitcast_u32<h2>((w & 0x000F000Fu) | e1024);
  const h2 q1 = bitcast_u32<h2>((w & 0x00F000F0u) | e64);
  const h2 q2 = bitcast_u32<h2>((hi & 0x000F000Fu) | e1024);
  const h2 q3 = bitcast_u32<h2>((hi & 0x00F000F0u) | e64);
  h2 d0 = q0 + zb_lo, d1 = q1 + zb_hi, d2 = q2 + zb_lo, d3 = q3 + zb_hi;
  if constexpr (kScaled) {
    d0 *= s2;
    d1 *= s2;
    d2 *= s2;
    d3 *= s2;
  }
  h8 out;
  out[0] = d0[0]; out[1] = d0[1]; out[2] = d1[0]; out[3] = d1[1];
  out[4] = d2[0]; out[5] = d2[1]; out[6] = d3[0]; out[7] = d3[1];
  return out;
}

}  // namespace glowq
