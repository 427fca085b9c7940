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

// g / (1 + e^-g) * u. The gate is divided first, as in every other form: g u may leave
// fp32 where the quotient is 0. A quarter of both, so that the reciprocal of the largest
// denominator is no denormal (which the instruction flushes); the quotient is put right
// by what it leaves, to within half an ulp as a division is, and where the denominator or
// the gate is infinite by div_fixup. At the end of a tile a wave alone on its SIMD waits
// for every instruction: 8192 rows of 28672 x 4096 1278 us (a division 1294, the bare
// reciprocal 1268), 2039 rows 341 (347, 341), 8 experts of 28672 x 4096 at 1024 rows 1631
// (1662, 1612).
DEVICE_INLINE float wt_silu(float g, float u) {
  const float d = __builtin_amdgcn_exp2f(__builtin_fmaf(g, -1.44269504f, -2.f)) + .25f;
  const float n = .25f * g, r = __builtin_amdgcn_rcpf(d), q = n * r;
  return __builtin_amdgcn_div_fixupf(
             __builtin_fmaf(__builtin_fmaf(-d, q, n), r, q), d, n) * u;
}

// A sum out of its accumulation register, in the order of the program: read where the
// compiler likes, all at once, they do not fit beside the operands of the next tile.
DEVICE_INLINE float wt_sum(float acc) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc));
  return v;
}

template <int I> using wt_int = std::integral_constant<int, I>;
