// Element types as f32, and packed int4 codes as fp16 integers: what every int4 product shares.
#pragma once

#include "krm_internal.h"

namespace krm {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

template <typename T>
__device__ inline float to_f32(T v);
template <>
__device__ inline float to_f32<float>(float v) { return v; }
template <>
__device__ inline float to_f32<__half>(__half v) { return __half2float(v); }
template <typename T>
__device__ inline T from_f32(float v);
template <>
__device__ inline float from_f32<float>(float v) { return v; }
template <>
__device__ inline __half from_f32<__half>(float v) { return __float2half_rn(v); }

// (a & mask) | bits in one VALU op: the compiler splits it in two when both constants are
// literals, because this ISA's three-operand encodings take no literal.
__device__ inline uint32_t and_or(uint32_t a, uint32_t mask, uint32_t bits) {
  uint32_t d;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "s"(mask), "v"(bits));
  return d;
}

// Eight codes of one u32 as four fp16 pairs holding the exact integers (u - 8): pair i = (code i,
// code i+4).  1024 + u is built in the fp16 mantissa, then the offset is removed with one packed op;
// codes in the upper nibble of a byte arrive as 1024 + 16u.  Two ops a pair, for activations stored in
// the same order.
__device__ inline void codes_to_half2(uint32_t word, half2_t (&q)[4]) {
  const uint32_t magic = 0x64006400u;  // (1024.0, 1024.0)
  const half2_t off_lo = {(_Float16)1032.0f, (_Float16)1032.0f};
  const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
  const half2_t off_hi = {(_Float16)-72.0f, (_Float16)-72.0f};
  const uint32_t upper = word >> 8;
  q[0] = __builtin_bit_cast(half2_t, and_or(word, 0x000F000Fu, magic)) - off_lo;
  q[1] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, and_or(word, 0x00F000F0u, magic)),
                                   sixteenth, off_hi);
  q[2] = __builtin_bit_cast(half2_t, and_or(upper, 0x000F000Fu, magic)) - off_lo;
  q[3] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, and_or(upper, 0x00F000F0u, magic)),
                                   sixteenth, off_hi);
}
// The same pairs as (u - 8) / 1024, exact, where the sum is multiplied by 1024 at the end: a code at the bottom
// of its half is the fp16 subnormal u 2^-24, one four bits up 16 u 2^-24, and one packed fma scales and offsets
// it.  Nine ops of which five take half the time of a packed one: a mask (v_and_b32, 2.4 clk a wave beside
// others, v_and_or_b32 4.4) needs no bits set beside it.
__device__ inline void codes_over_1024(uint32_t word, half2_t (&q)[4]) {
  const half2_t low = {(_Float16)16384.0f, (_Float16)16384.0f}, high = {(_Float16)1024.0f, (_Float16)1024.0f};
  const half2_t offset = {(_Float16)-0.0078125f, (_Float16)-0.0078125f};
  const uint32_t upper = word >> 8;
  q[0] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, word & 0x000F000Fu), low, offset);
  q[1] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, word & 0x00F000F0u), high, offset);
  q[2] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, upper & 0x000F000Fu), low, offset);
  q[3] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, upper & 0x00F000F0u), high, offset);
}
// Sums over K that stay 1024 times smaller until their end reach subnormal numbers 1024 times sooner: an fp16 scale
// or result is far from there, an f32 scale beside an f32 result need not be.  There a group's scale is multiplied
// by 1024, unless one of the wave's would leave f32's range by that: then (what is returned) its sums are, where they
// are.
template <int N>
__device__ inline bool scales_whole(float (&scale)[N]) {
  uint64_t past = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) past |= __builtin_amdgcn_ballot_w64(fabsf(scale[i]) >= 0x1p117f);
  const float factor = past ? 1.0f : 1024.0f;
#pragma unroll
  for (int i = 0; i < N; ++i) scale[i] *= factor;
  return past != 0;
}
// Eight consecutive fp16 activations (x0..x7 in four dwords) regrouped to match
// codes_to_half2: pair i = (x_i, x_{i+4}).
__device__ inline void pair_activations(const uint4& raw, half2_t (&p)[4]) {
  p[0] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(raw.z, raw.x, 0x05040100u));
  p[1] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(raw.z, raw.x, 0x07060302u));
  p[2] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(raw.w, raw.y, 0x05040100u));
  p[3] = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(raw.w, raw.y, 0x07060302u));
}

// The same as one operand of a matrix instruction: (c0,c4,c1,c5,c2,c6,c3,c7), each (u - 8) / 1024 or (OVER false)
// whole.
template <bool OVER>
__device__ inline half8_t ints_paired(uint32_t word) {
  half2_t q[4];
  if constexpr (OVER) codes_over_1024(word, q); else codes_to_half2(word, q);
  return half8_t{q[0].x, q[0].y, q[1].x, q[1].y, q[2].x, q[2].y, q[3].x, q[3].y};
}

}  // namespace
}  // namespace krm
