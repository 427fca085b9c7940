// Common device helpers for gpustack_amd CDNA4 (gfx950 / MI355X) kernels.
//
// Design notes (MI355X-first):
//  - wavefront = 64 lanes; all cross-lane idioms use 64-wide shuffles.
//  - bf16 is the serving dtype; all reductions accumulate in f32.
//  - memory-bound kernels vectorize loads as 16 B/lane (u16x8 for bf16).
#pragma once

#include <hip/hip_fp8.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#define WAVE_SIZE 64
#define DEVICE_INLINE __device__ __forceinline__

typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
typedef __attribute__((ext_vector_type(4))) unsigned short u16x4;
typedef __attribute__((ext_vector_type(8))) unsigned short u16x8;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) float f32x8;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

// bf16 (stored as unsigned short) <-> f32
__device__ __forceinline__ float bf2f(unsigned short u) {
  union { float f; unsigned int i; } v;
  v.i = ((unsigned int)u) << 16;
  return v.f;
}

// round-to-nearest-even f32 -> bf16: v_cvt_pk_bf16_f32, for every number the bits that
// adding half and cutting gave (all 2^32 compared; one that is none stays none), in one
// instruction for two of them instead of seven for one (a prompt of 7999 rows 11711 ->
// 11639 us; short steps gain less than they spread).
__device__ __forceinline__ unsigned short f2bf(float f) {
  return __builtin_bit_cast(unsigned short, (__bf16)f);
}

typedef __attribute__((ext_vector_type(8))) unsigned char u8x8;
typedef __attribute__((ext_vector_type(4))) unsigned char u8x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

// OCP fp8 e4m3 (gfx950-native v_cvt_f32_fp8 / v_cvt_pk_fp8_f32)
__device__ __forceinline__ float fp8_to_f32(unsigned char u) {
  __hip_fp8_e4m3 v;
  v.__x = u;
  return (float)v;
}

__device__ __forceinline__ unsigned char f32_to_fp8(float f) {
  __hip_fp8_e4m3 v(f);
  return v.__x;
}

__device__ __forceinline__ void fp8x8_to_f32(const u8x8 v, float* out) {
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = fp8_to_f32(v[i]);
}

__device__ __forceinline__ void bf8_to_f32(const u16x8 v, float* out) {
#pragma unroll
  for (int i = 0; i < 8; ++i) out[i] = bf2f(v[i]);
}

__device__ __forceinline__ u16x8 f32_to_bf8(const float* in) {
  u16x8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = f2bf(in[i]);
  return v;
}

// Eight neighbours of a product cut over k: fp32 parts `stride` apart, added up in
// their order and rounded, as the product's own join does it. Four parts are in
// flight at a time, or eight where there are more: what adds a few rows up waits for
// the memory once or twice and does little else.
template <int U>
DEVICE_INLINE void add_parts8(float* sum, const float* p, long stride, int parts) {
  for (int s0 = 0; s0 < parts; s0 += U) {
    f32x4 v[U][2];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const float* at = p + min(s0 + i, parts - 1) * stride;
      v[i][0] = *reinterpret_cast<const f32x4*>(at);
      v[i][1] = *reinterpret_cast<const f32x4*>(at + 4);
    }
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (s0 + i < parts)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          sum[j] = s0 + i == 0 ? v[0][j / 4][j % 4] : sum[j] + v[i][j / 4][j % 4];
  }
}
DEVICE_INLINE u16x8 join_parts8(const float* p, long stride, int parts) {
  float sum[8];
  if (parts > 4) add_parts8<8>(sum, p, stride, parts);
  else add_parts8<4>(sum, p, stride, parts);
  return f32_to_bf8(sum);
}

// Eight neighbours of k bf16 rows `stride` apart, added up in fp32 in their order and
// rounded. Four rows are in flight at a time.
DEVICE_INLINE u16x8 sum_rows8(const unsigned short* p, long stride, int k) {
  float sum[8];
  for (int j0 = 0; j0 < k; j0 += 4) {
    u16x8 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      v[i] = *reinterpret_cast<const u16x8*>(p + min(j0 + i, k - 1) * stride);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f[8];
      bf8_to_f32(v[i], f);
      if (j0 + i < k)
#pragma unroll
        for (int j = 0; j < 8; ++j) sum[j] = j0 + i == 0 ? f[j] : sum[j] + f[j];
    }
  }
  return f32_to_bf8(sum);
}

// A value and that of the lane 32 (M = 32) or 16 away, in either order, without the
// LDS. The two operands of the swap are kept apart: given one value twice the compiler
// takes both results for the same.
template <int M>
DEVICE_INLINE f32x2 with_lane(float v) {
  const unsigned int a = __builtin_bit_cast(unsigned int, v);
  unsigned int b = a;
  asm("" : "+v"(b));
  const auto r = M == 16 ? __builtin_amdgcn_permlane16_swap(a, b, false, false)
                         : __builtin_amdgcn_permlane32_swap(a, b, false, false);
  const unsigned int x = r[0], y = r[1];
  return f32x2{__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
}

// The value of the lane N places on in a row of 16 lanes, around its end.
template <int N>
DEVICE_INLINE float row_turned(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N,
                                         0xf, 0xf, true));
}

// Full-wave (64-lane) reductions, in the order and to the bit of a butterfly (lanes 32,
// 16, 8, 4, 2, 1 apart; once lanes 2 N apart agree, N on and N apart are the same), but
// not through the LDS, whose six exchanges are most of a microsecond in a row kernel.
__device__ __forceinline__ float wave_reduce_sum(float x) {
  f32x2 p = with_lane<32>(x);
  p = with_lane<16>(p[0] + p[1]);
  x = p[0] + p[1];
  x += row_turned<8>(x);
  x += row_turned<4>(x);
  x += row_turned<2>(x);
  return x + row_turned<1>(x);
}

__device__ __forceinline__ float wave_reduce_max(float x) {
  f32x2 p = with_lane<32>(x);
  p = with_lane<16>(fmaxf(p[0], p[1]));
  x = fmaxf(p[0], p[1]);
  x = fmaxf(x, row_turned<8>(x));
  x = fmaxf(x, row_turned<4>(x));
  x = fmaxf(x, row_turned<2>(x));
  return fmaxf(x, row_turned<1>(x));
}

// Maximum of a lane and lane ^ 32, in all lanes.
DEVICE_INLINE float half_wave_max(float x) {
  const f32x2 p = with_lane<32>(x);
  return fmaxf(p[0], p[1]);
}

// Reduction across a 16-lane subgroup (lanes with equal l>>4).
__device__ __forceinline__ float group16_reduce_sum(float x) {
  x += row_turned<8>(x);
  x += row_turned<4>(x);
  x += row_turned<2>(x);
  return x + row_turned<1>(x);
}

// n / (1 + e^-z): SiLU (n = z) and the sigmoid (n = 1) of row kernels, whose time they
// are. The power of two of z log2 e; what is left of that product's rounding, and what
// the denominator's sum rounded away, go to the remainder that puts the quotient right,
// so that little but the power's own error stays. 2048 x 256 x 2048 of them 605 us where
// expf and a division are 757. Norm of the error of 4 M normal z 2.64e-8 (expf and a
// division 3.94e-8), of z in -20 .. 20 2.32e-8 (3.30e-8), the largest, down to results
// that leave fp32, 1.34e-7 of the result (1.79e-7). A quarter of both sides, since the
// reciprocal of the largest denominator is no denormal then.
DEVICE_INLINE float over_one_plus_exp(float n, float z) {
  const float h = z * -1.44269504f;
  const float e = .25f * __builtin_amdgcn_exp2f(h);
  const float l = __builtin_fmaf(z, -1.92596303e-8f, __builtin_fmaf(z, -1.44269504f, -h));
  const float d = e + .25f;
  const float lost = fminf(e, .25f) - (d - fmaxf(e, .25f));
  // an infinite z has no product to put right, an infinite denominator needs nothing
  const float g = __builtin_fabsf(h) < 128.f ? __builtin_fmaf(e, l * 0.693147181f, lost) : 0.f;
  const float m = .25f * n, r = __builtin_amdgcn_rcpf(d), q = m * r;
  return __builtin_amdgcn_div_fixupf(
      __builtin_fmaf(__builtin_fmaf(-g, q, __builtin_fmaf(-d, q, m)), r, q), d, m);
}

// Loads from memory straight to LDS address `to` + 16 * lane, 16 bytes a lane,
// from base + off bytes or from `at`; addresses are multiples of 16. Inline asm,
// because the compiler puts a wait for all such loads of its builtin in front of
// LDS reads that it cannot tell from them. They write no register but m0, which
// the compiler is told; the kernel waits for them itself (s_waitcnt vmcnt, then its
// barrier).
DEVICE_INLINE unsigned int lds_address(const unsigned short* p) {
  return (unsigned int)(unsigned long)(
      const __attribute__((address_space(3))) unsigned short*)p;
}
// (m0 is reserved, which clang warns about where it is named as written to.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
DEVICE_INLINE void load_to_lds(const unsigned short* base, unsigned int off,
                               const unsigned short* to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               ::"s"(lds_address(to)), "v"(off), "s"(base) : "m0", "memory");
}
DEVICE_INLINE void load_to_lds(const unsigned short* at,
                               const unsigned short* to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               ::"s"(lds_address(to)), "v"(at) : "m0", "memory");
}
#pragma clang diagnostic pop

#define HIP_CHECK_KERNEL()                                        \
  do {                                                            \
    hipError_t e_ = hipGetLastError();                            \
    if (e_ != hipSuccess) {                                       \
      TORCH_CHECK(false, "HIP kernel launch failed: ",            \
                  hipGetErrorString(e_));                         \
    }                                                             \
  } while (0)

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
