// Products with packed int4 weights for MI355X (gfx950): out[M, N] =
// x[M, K] W^T with W kept packed in HBM, and the transient expansion to bf16
// that prompt-sized products use in front of the library GEMM.
//
// Packed layout (models/quantized.py pack_w4_runtime): qw u8 [N, K/2] in
// FRAGMENT ORDER — within each 128-k block, the 16 bytes lane group lg loads
// hold exactly the 32 nibbles (4 MFMA k-chunks x 8 values) of its operand
// fragments:
//   nibble i (0..31) of lg's 16 bytes = q[row][blk*128 + (i/8)*32 + lg*8 + i%8]
// Scales / zero-scales: bf16 [N, K/128], one group per 128-k block.
// w = q * s - zs   (zs = zero * s, precomputed).
//
// Few rows (decode). A workgroup of 8 or 16 waves owns 16 NTW columns of up to
// 64 rows; its waves take the k blocks in turn (neighbouring blocks of a row
// are read together) and meet in the LDS at the end, so no second kernel and
// no partial results in memory.
//  - A nibble becomes bf16 without arithmetic: 0x4300 | q is 128 + q, two at
//    a time (q_j beside q_{j+4}; x fragments are put in the same order with
//    four v_perm). The products of a block are exact in q; its scale and
//    offset are applied to the fp32 sums:
//      out += s * (x . (128 + q)) - (128 s + zs) * sum(x),
//    sum(x) coming from one more product with a fragment of ones, shared by
//    the NTW column tiles. The weights are never rounded to bf16 here, as the
//    expansion does.
//  - 16-byte weight loads run one block ahead; scales are staged in the LDS.
// Bound by the weight stream (0.5 bytes a weight).
#include "common.h"

namespace {

constexpr int W4_KC = 128;

typedef __attribute__((ext_vector_type(8))) short w4_s16x8;

DEVICE_INLINE f32x4 w4_mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(w4_s16x8, a), __builtin_bit_cast(w4_s16x8, b), c, 0, 0, 0);
}

// eight nibbles as bf16 128 + q in the order 0 4 1 5 2 6 3 7
DEVICE_INLINE u32x4 w4_bf16(unsigned int d) {
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    o[j] = ((d >> (4 * j)) & 0x000f000fu) | 0x43004300u;
  return o;
}

// eight bf16 in that order
DEVICE_INLINE u32x4 w4_order(u32x4 v) {
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    o[2 * j] = __builtin_amdgcn_perm(v[2 + j], v[j], 0x05040100u);
    o[2 * j + 1] = __builtin_amdgcn_perm(v[2 + j], v[j], 0x07060302u);
  }
  return o;
}

template <int MT, int NTW, int WAVES>
__global__ __launch_bounds__(WAVES * WAVE_SIZE) void w4_rows_kernel(
    unsigned short* __restrict__ out,       // [M, N] bf16
    const unsigned short* __restrict__ x,   // [M, K] bf16
    const unsigned char* __restrict__ qw,   // [N, K/2] frag-ordered nibbles
    const unsigned short* __restrict__ sc,  // [N, K/128] bf16 scale
    const unsigned short* __restrict__ zs,  // [N, K/128] bf16 zero*scale
    int M, int N, int K) {
  constexpr int COLS = 16 * NTW, ROWS = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) float w4_lds[];
  const int nb = K / W4_KC;
  // scales of the workgroup's columns, [nb][COLS] (s low half, zs high), then
  // the waves' partial sums [8][ROWS][COLS]
  unsigned int* sz = reinterpret_cast<unsigned int*>(w4_lds);

  const int m0 = blockIdx.y * ROWS;
  const int n0 = blockIdx.x * COLS;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lc = lane & 15;
  const int lg = lane >> 4;

  const unsigned char* wp[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t)
    wp[t] = qw + (long)(n0 + t * 16 + lc) * (K / 2) + lg * 16;
  const unsigned short* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    xp[t] = x + (long)min(m0 + t * 16 + lc, M - 1) * K + lg * 8;

  // block numbers start at the workgroup's own place in the row: rows lie a
  // power of two apart, and workgroups that all read the same columns of
  // their rows would meet on a few memory channels
  const int rot = blockIdx.x % nb;
  auto block = [&](int b) { return b + rot < nb ? b + rot : b + rot - nb; };
  u32x4 wc[NTW], wn[NTW];
  const int b0 = block(min(wave, nb - 1));
#pragma unroll
  for (int t = 0; t < NTW; ++t)
    wc[t] = *reinterpret_cast<const u32x4*>(wp[t] + (long)b0 * 64);

  for (int u = tid; u < COLS * nb; u += WAVES * WAVE_SIZE) {
    const int c = u / nb, b = u % nb;
    const long at = (long)(n0 + c) * nb + b;
    sz[b * COLS + c] = (unsigned int)sc[at] | ((unsigned int)zs[at] << 16);
  }
  __syncthreads();

  f32x4 acc[MT][NTW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NTW; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};

  auto multiply = [&](int b) {
    u32x4 xa[MT][4];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        xa[i][c] = w4_order(*reinterpret_cast<const u32x4*>(
            xp[i] + b * W4_KC + c * 32));
    f32x4 xs[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      xs[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) xs[i] = w4_mfma(xa[i][c], ones, xs[i]);
    }
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      f32x4 p[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) p[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const u32x4 wf = w4_bf16(wc[t][c]);
#pragma unroll
        for (int i = 0; i < MT; ++i) p[i] = w4_mfma(xa[i][c], wf, p[i]);
      }
      const unsigned int v = sz[b * COLS + t * 16 + lc];
      const float s = __builtin_bit_cast(float, v << 16);
      const float z = 128.f * s + __builtin_bit_cast(float, v & 0xffff0000u);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[i][t][r] += s * p[i][r] - z * xs[i][r];
    }
  };
  int j = wave;
  for (; j + WAVES < nb; j += WAVES) {
    const long bn = (long)block(j + WAVES) * 64;
#pragma unroll
    for (int t = 0; t < NTW; ++t)
      wn[t] = *reinterpret_cast<const u32x4*>(wp[t] + bn);
    multiply(block(j));
#pragma unroll
    for (int t = 0; t < NTW; ++t) wc[t] = wn[t];
  }
  if (j < nb) multiply(block(j));

  __syncthreads();                       // the scales are done with
  // D[row = lg*4 + r][col = lc] per 16x16 tile
  float* red = w4_lds;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(wave * ROWS + i * 16 + lg * 4 + r) * COLS + t * 16 + lc] =
            acc[i][t][r];
  __syncthreads();
  for (int u = tid; u < ROWS * COLS; u += WAVES * WAVE_SIZE) {
    const int row = m0 + u / COLS;
    if (row >= M) break;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) v += red[w * ROWS * COLS + u];
    out[(long)row * N + n0 + u % COLS] = f2bf(v);
  }
}

// Transient dequant for prefill-shaped GEMMs (bandwidth-bound): packed
// frag-order nibbles -> bf16 [N, K] in canonical k order, so hipBLASLt
// consumes the result directly. Each thread expands one 16-byte packed
// chunk (lane-lg slice of a 128-k block) into its four 8-value octets at
// k = blk*128 + c*32 + lg*8.
__global__ __launch_bounds__(256) void w4_dequant_kernel(
    unsigned short* __restrict__ out,      // [N, K] bf16
    const unsigned char* __restrict__ qw,  // [N, K/2] frag-ordered
    const unsigned short* __restrict__ sc, // [N, K/128]
    const unsigned short* __restrict__ zs, // [N, K/128]
    long N, int K) {
  const long chunks = N * (K / 32);        // 16B packed chunks
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < chunks;
       idx += (long)gridDim.x * blockDim.x) {
    const long row = idx / (K / 32);
    const int ck = idx % (K / 32);         // chunk within row
    const int blk = ck / 4;
    const int lg = ck % 4;
    const uint4 w = *reinterpret_cast<const uint4*>(
        qw + row * (K / 2) + (long)blk * 64 + lg * 16);
    const float s = bf2f(sc[row * (K / 128) + blk]);
    const float z = bf2f(zs[row * (K / 128) + blk]);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const unsigned int d = (&w.x)[c];
      unsigned short o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = f2bf((float)((d >> (4 * j)) & 0xF) * s - z);
      *reinterpret_cast<u16x8*>(out + row * K + blk * 128 + c * 32 + lg * 8) =
          *reinterpret_cast<u16x8*>(o);
    }
  }
}

}  // namespace

void w4_dequant_launch(void* out, const void* qw, const void* sc,
                       const void* zs, long N, int K, int* err_unsupported,
                       hipStream_t s) {
  *err_unsupported = 0;
  if (K % W4_KC != 0) { *err_unsupported = 1; return; }
  const long chunks = N * (K / 32);
  long grid = (chunks + 255) / 256;
  if (grid > 16384) grid = 16384;
  hipLaunchKernelGGL(w4_dequant_kernel, dim3((unsigned)grid), dim3(256), 0, s,
                     (unsigned short*)out, (const unsigned char*)qw,
                     (const unsigned short*)sc, (const unsigned short*)zs, N,
                     K);
}

namespace {
template <int MT, int NTW, int WAVES>
void w4_rows(void* out, const void* x, const void* qw, const void* sc,
             const void* zs, int M, int N, int K, hipStream_t s) {
  const size_t scales = (size_t)(K / W4_KC) * 16 * NTW * 4;
  const size_t sums = (size_t)WAVES * 16 * MT * 16 * NTW * 4;
  hipLaunchKernelGGL((w4_rows_kernel<MT, NTW, WAVES>),
                     dim3(N / (16 * NTW), (M + 16 * MT - 1) / (16 * MT)),
                     dim3(WAVES * WAVE_SIZE), scales > sums ? scales : sums, s,
                     (unsigned short*)out, (const unsigned short*)x,
                     (const unsigned char*)qw, (const unsigned short*)sc,
                     (const unsigned short*)zs, M, N, K);
}
}  // namespace

// The form by columns: workgroups of four column tiles per wave (two at 64
// rows) from 448 of them on; of two from 160 on, with 16 waves while x is one
// row tile (6144 x 4096, us at 16 rows: 9.1 against 12.3 with one tile, at 64
// rows 21.5 against 33.7); else of one, which keeps every CU on the stream
// (4096 x 4096 at 16 rows: 7.6 against 8.7 with two), with 16 waves for long
// rows (4096 x 14336 at one row: 11.9 against 14.5). The scales of K / 128
// blocks stay under 64 KB.
void w4_gemm_launch(void* out, const void* x, const void* qw, const void* sc,
                    const void* zs, int M, int N, int K,
                    int* err_unsupported, hipStream_t s) {
  *err_unsupported = 0;
  if (N % 64 != 0 || K % W4_KC != 0 || K / W4_KC > 1024) {
    *err_unsupported = 1;
    return;
  }
  if (M == 0) return;
  const int nb = K / W4_KC;
  const int ntw = N / 64 >= 448 && nb <= 256 ? 4
                  : N / 32 >= 160 && nb <= 512 ? 2 : 1;
#define W4_ARGS out, x, qw, sc, zs, M, N, K, s
#define W4_ROWS(MT)                                                          \
  do {                                                                       \
    if (ntw == 4) w4_rows<MT, (MT) == 4 ? 2 : 4, 8>(W4_ARGS);                \
    else if (ntw == 2) w4_rows<MT, 2, (MT) == 1 ? 16 : 8>(W4_ARGS);          \
    else if (nb >= 64 && (MT) <= 2) w4_rows<MT, 1, (MT) <= 2 ? 16 : 8>(W4_ARGS); \
    else w4_rows<MT, 1, 8>(W4_ARGS);                                         \
  } while (0)
  if (M <= 16) W4_ROWS(1);
  else if (M <= 32) W4_ROWS(2);
  else W4_ROWS(4);
#undef W4_ARGS
#undef W4_ROWS
}
