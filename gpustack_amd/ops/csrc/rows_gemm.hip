// Decode products for MI355X (gfx950): out[M, N] = x[M, K] W^T in bf16 for up
// to 64 rows, fp32 sums.
//
// A workgroup of 8 waves owns 16 NTW columns; its waves take the 128-k blocks
// of those weight rows in turn and meet in the LDS at the end, so a product of
// few columns still has every wave of the chip on the weight stream, with no
// partial results in memory and no second kernel. A weight row's 16-byte
// chunks are the MFMA operand as they lie; one block of them is in flight while
// the block before is multiplied. x comes from the L2.
// Bound by the weight stream (2 bytes a weight), and for more than 32 rows by
// x out of the L2: each workgroup reads all of it.
#include "common.h"

namespace {

constexpr int RG_KC = 128;
constexpr int RG_WAVES = 8;
constexpr int RG_THREADS = RG_WAVES * WAVE_SIZE;

typedef __attribute__((ext_vector_type(8))) short rg_s16x8;

template <int MT, int NTW>
__global__ __launch_bounds__(RG_THREADS) void rows_gemm_kernel(
    unsigned short* __restrict__ out,       // [M, N]
    const unsigned short* __restrict__ x,   // [M, K], row stride xs
    const unsigned short* __restrict__ w,   // [N, K]
    int M, int N, int K, long xs) {
  constexpr int COLS = 16 * NTW, ROWS = 16 * MT;
  __shared__ float red[RG_WAVES * ROWS * COLS];
  const int nb = K / RG_KC;
  const int n0 = blockIdx.x * COLS;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lc = lane & 15;
  const int lg = lane >> 4;

  const unsigned short* wp[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t)
    wp[t] = w + (long)min(n0 + t * 16 + lc, N - 1) * K + lg * 8;
  const unsigned short* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
    xp[t] = x + (long)min(t * 16 + lc, M - 1) * xs + lg * 8;

  // Block numbers start at the workgroup's own place in the row: rows lie a
  // power of two apart, and workgroups that all read the same columns of
  // their rows would meet on a few memory channels.
  const int rot = blockIdx.x % nb;
  auto block = [&](int b) { return b + rot < nb ? b + rot : b + rot - nb; };
  u32x4 wc[NTW][4], wn[NTW][4];
  const int b0 = block(min(wave, nb - 1));
#pragma unroll
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      wc[t][c] = *reinterpret_cast<const u32x4*>(wp[t] + b0 * RG_KC + c * 32);

  f32x4 acc[MT][NTW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int t = 0; t < NTW; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&](int b) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      u32x4 xa[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        xa[m] = *reinterpret_cast<const u32x4*>(xp[m] + b * RG_KC + c * 32);
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(rg_s16x8, xa[m]),
              __builtin_bit_cast(rg_s16x8, wc[t][c]), acc[m][t], 0, 0, 0);
    }
  };
  int i = wave;
  for (; i + RG_WAVES < nb; i += RG_WAVES) {
    const int bn = block(i + RG_WAVES);
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        wn[t][c] = *reinterpret_cast<const u32x4*>(wp[t] + bn * RG_KC + c * 32);
    multiply(block(i));
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c) wc[t][c] = wn[t][c];
  }
  if (i < nb) multiply(block(i));

  // D[row = lg*4 + r][col = lc] per 16x16 tile
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NTW; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        red[(wave * ROWS + m * 16 + lg * 4 + r) * COLS + t * 16 + lc] =
            acc[m][t][r];
  __syncthreads();
  for (int u = tid; u < ROWS * COLS; u += RG_THREADS) {
    const int row = u / COLS, col = n0 + u % COLS;
    if (row >= M || col >= N) continue;
    float v = 0.f;
#pragma unroll
    for (int w8 = 0; w8 < RG_WAVES; ++w8) v += red[w8 * ROWS * COLS + u];
    out[(long)row * N + col] = f2bf(v);
  }
}

template <int MT, int NTW>
void rows_gemm(void* out, const void* x, const void* w, int M, int N, int K,
               long xs, hipStream_t s) {
  hipLaunchKernelGGL((rows_gemm_kernel<MT, NTW>),
                     dim3((N + 16 * NTW - 1) / (16 * NTW)), dim3(RG_THREADS),
                     0, s, (unsigned short*)out, (const unsigned short*)x,
                     (const unsigned short*)w, M, N, K, xs);
}

}  // namespace

void rows_gemm_launch(void* out, const void* x, const void* w, int M, int N,
                      int K, long xs, int* err_unsupported, hipStream_t s) {
  *err_unsupported = K % RG_KC != 0 || K == 0 || M > 64;
  if (*err_unsupported || M == 0 || N == 0) return;
  const bool wide = N / 32 >= 512;
  if (M <= 16) {
    if (wide) rows_gemm<1, 2>(out, x, w, M, N, K, xs, s);
    else rows_gemm<1, 1>(out, x, w, M, N, K, xs, s);
  } else if (M <= 32) {
    if (wide) rows_gemm<2, 2>(out, x, w, M, N, K, xs, s);
    else rows_gemm<2, 1>(out, x, w, M, N, K, xs, s);
  } else {
    if (wide) rows_gemm<4, 2>(out, x, w, M, N, K, xs, s);
    else rows_gemm<4, 1>(out, x, w, M, N, K, xs, s);
  }
}
