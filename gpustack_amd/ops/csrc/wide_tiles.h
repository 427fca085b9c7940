// What the kernels of one wave a SIMD share: descriptors for loads that end at their
// operand's edge, sums out of the accumulation registers.
#pragma once

#include "common.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(4))) int i32x4;

DEVICE_INLINE unsigned wt_pack(float lo, float hi) {
  const f32x2 v{lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// Descriptor of `bytes` bytes at p; loads beyond them bring no memory.
DEVICE_INLINE i32x4 wt_rsrc(const void* p, unsigned bytes) {
  const unsigned long a = (unsigned long)p;
  return i32x4{(int)a, (int)(a >> 32) & 0xffff, (int)bytes, 0x00020000};
}

// The gate is divided first, as in every other form: g * u may leave fp32 where the
// quotient is 0. A division costs the end of a tile nothing that shows (8192 rows of
// 28672 x 4096 1254 us, with the reciprocal 1254).
DEVICE_INLINE float wt_silu(float g, float u) { return g / (1.f + __expf(-g)) * u; }

// A sum out of its accumulation register, in the order of the program: read where the
// compiler likes, all at once, they do not fit beside the operands of the next tile.
DEVICE_INLINE float wt_sum(float acc) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc));
  return v;
}

template <int I> using wt_int = std::integral_constant<int, I>;
