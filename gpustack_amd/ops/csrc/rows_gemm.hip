// Decode products for MI355X (gfx950): out[M, N] = x[M, K] W^T in bf16 for few
// rows, fp32 sums: up to 16 without a tile, up to 128 with one (below).
//
// A workgroup of 8 waves owns 16 NTW columns; its waves take the 128-k blocks
// of those weight rows in turn and meet in the LDS at the end, so a product of
// few columns still has every wave of the chip on the weight stream, with no
// partial results in memory and no second kernel. A weight row's 16-byte
// chunks are the MFMA operand as they lie; one block of them is in flight while
// the block before is multiplied. x comes from the L2.
// Bound by the weight stream (2 bytes a weight): 65536 x 4096 at one row 88 us
// (6.1 TB/s), 4096 x 4096 9.5, which is latency.
#include "common.h"

namespace {

constexpr int RG_KC = 128;
constexpr int RG_WAVES = 8;
constexpr int RG_THREADS = RG_WAVES * WAVE_SIZE;

typedef __attribute__((ext_vector_type(8))) short rg_s16x8;

template <int NTW>
__global__ __launch_bounds__(RG_THREADS) void rows_gemm_kernel(
    unsigned short* __restrict__ out,       // [M, N]
    const unsigned short* __restrict__ x,   // [M, K], row stride xs
    const unsigned short* __restrict__ w,   // [N, K]
    int M, int N, int K, long xs) {
  constexpr int COLS = 16 * NTW, ROWS = 16;
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
  const unsigned short* xp = x + (long)min(lc, M - 1) * xs + lg * 8;

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

  f32x4 acc[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto multiply = [&](int b) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const u32x4 xa =
          *reinterpret_cast<const u32x4*>(xp + b * RG_KC + c * 32);
#pragma unroll
      for (int t = 0; t < NTW; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(rg_s16x8, xa),
            __builtin_bit_cast(rg_s16x8, wc[t][c]), acc[t], 0, 0, 0);
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
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[(wave * ROWS + lg * 4 + r) * COLS + t * 16 + lc] = acc[t][r];
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

// Up to 128 rows. Reading x beside every 16 weight rows, as above, would ask
// the L2 for up to eight times the weights, so here 4 waves share a tile of
// 16 MT rows and 16 NT columns: both sides of a 64-k step go to a ring of S
// buffers in the LDS, S - 1 steps ahead of the products, which is what keeps
// HBM busy from two workgroups a CU. A step waits only for its own buffer, and
// its barrier frees the buffer that the new step is loaded into.
// Rows of 128 bytes; the 16-byte chunk c of row r lies at c ^ (r / 2 % 8), free
// of conflicts for 16 rows of one chunk. Weights are the A operand, so a lane
// ends with 4 neighbouring columns of a row. Few columns are cut over k as
// well, into fp32 parts that rows_join_kernel adds up.
// More than 128 rows are row tiles of their own, always in parts. (Row tiles of a
// piece of the weights one behind the other on an XCD, for its L2, lost: 512 rows
// of 4096 x 14336 64 -> 77 us; one behind the other in time the Infinity Cache
// serves them, and 4 or 8 parts leave an XCD a quarter or less of x.)
// Bound by the weight stream: 28672 x 4096 at 48 rows 41 us (5.7 TB/s; the
// library 51), 4096 x 14336 in four
// parts 26 with the join (36), 128256 x 4096 182 (254). One workgroup a CU
// takes the LDS for a deeper ring: 28672 x 4096 at 96 rows 61 -> 46.
constexpr int RT_K = 64;

template <int L>
DEVICE_INLINE void rt_wait(int ahead) {      // all but `ahead` steps are there
  if (ahead >= 6) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(6 * L) : "memory");
  else if (ahead == 5) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(5 * L) : "memory");
  else if (ahead == 4) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(4 * L) : "memory");
  else if (ahead == 3) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(3 * L) : "memory");
  else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * L) : "memory");
  else if (ahead == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(L) : "memory");
  else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// SILU: w holds N gate rows and N up rows, and out [M, N] is silu(gate) * up of
// the fp32 sums; a wave's column tiles are half gate, half up, so that a lane
// has both of a column. That saves the activation's launch and the wide row's
// rounding: 64 rows of 16384 x 2048 18.8 + 4.9 -> 17.3 us, 48 of 28672 x 4096
// 42.2 + 5.0 -> 44.1, one 40.5 + 4.6 -> 42.8.
enum RowsOut { ROWS, SPLIT_K, SILU };

template <int MT, int NT, int S, int OUT>
__global__ __launch_bounds__(256, 2) void rows_tile_kernel(
    void* __restrict__ out,                 // bf16 [M, N] or fp32 [splits, M, N]
    const unsigned short* __restrict__ x,   // [M, K], row stride xs
    const unsigned short* __restrict__ w,   // [N, K]
    int M, int N, int K, long xs, int splits) {
  constexpr bool SPLIT = OUT == SPLIT_K;
  constexpr int CT = OUT == SILU ? 8 * NT : 16 * NT;  // columns of a tile
  static_assert(OUT != SILU || NT % 4 == 0, "pairs of tiles");
  constexpr int BUF = 16 * (MT + NT) * RT_K;
  constexpr int L = (MT + NT) / 2;          // loads of a wave in a step
  static_assert(S >= 2 && S <= 8 && 6 * L <= 63, "the waits above");
  __shared__ unsigned short lds[S * BUF];
  const int split = SPLIT ? blockIdx.x % splits : 0;
  const int n0 = (SPLIT ? blockIdx.x / splits : blockIdx.x) * CT;
  const int m0 = blockIdx.y * 16 * MT;
  const int total = K / RT_K;
  const int from = SPLIT ? (int)((long)total * split / splits) : 0;
  const int n = (SPLIT ? (int)((long)total * (split + 1) / splits) : total) - from;
  const int tid = threadIdx.x;
  const int lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave >> 1, wn = wave & 1;
  const int lc = lane & 15, lg = lane >> 4;

  // a wave instruction fills 8 rows; wave w takes every fourth of them
  const unsigned short* xp[MT / 2];
  const unsigned short* wp[NT / 2];
#pragma unroll
  for (int i = 0; i < MT / 2; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    xp[i] = x + (long)min(m0 + row, M - 1) * xs +
            ((lane & 7) ^ ((row >> 1) & 7)) * 8;
  }
#pragma unroll
  for (int i = 0; i < NT / 2; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    long col;
    if constexpr (OUT == SILU) {             // a wave's rows: 4 NT gate, 4 NT up
      const int local = row % (8 * NT);
      col = min(n0 + row / (8 * NT) * 4 * NT + local % (4 * NT), N - 1) +
            (local >= 4 * NT ? (long)N : 0l);
    } else {
      col = min(n0 + row, N - 1);
    }
    wp[i] = w + col * K + ((lane & 7) ^ ((row >> 1) & 7)) * 8;
  }
  // first steps differ from workgroup to workgroup, as above
  const int rot = blockIdx.x % n;
  auto stage = [&](int i) {
    const int k0 = (from + (i + rot < n ? i + rot : i + rot - n)) * RT_K;
    unsigned short* d = lds + i % S * BUF + wave * 8 * RT_K;
#pragma unroll
    for (int j = 0; j < MT / 2; ++j)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) unsigned int*)(xp[j] + k0),
          (__attribute__((address_space(3))) unsigned int*)(d + j * 32 * RT_K),
          16, 0, 0);
#pragma unroll
    for (int j = 0; j < NT / 2; ++j)
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) unsigned int*)(wp[j] + k0),
          (__attribute__((address_space(3))) unsigned int*)(
              d + (16 * MT + j * 32) * RT_K),
          16, 0, 0);
  };

  f32x4 acc[MT / 2][NT / 2];
#pragma unroll
  for (int m = 0; m < MT / 2; ++m)
#pragma unroll
    for (int t = 0; t < NT / 2; ++t) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (i < n) stage(i);
  for (int i = 0; i < n; ++i) {
    rt_wait<L>(min(S - 2, n - 1 - i));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (i + S - 1 < n) stage(i + S - 1);
    const unsigned short* xl = lds + i % S * BUF + wm * MT / 2 * 16 * RT_K;
    const unsigned short* wl =
        lds + i % S * BUF + (MT + wn * NT / 2) * 16 * RT_K;
#pragma unroll
    for (int c = 0; c < RT_K / 32; ++c) {
      const int at = lc * RT_K + ((c * 4 + lg) ^ ((lc >> 1) & 7)) * 8;
      u32x4 fx[MT / 2], fw[NT / 2];
#pragma unroll
      for (int t = 0; t < NT / 2; ++t)
        fw[t] = *reinterpret_cast<const u32x4*>(wl + t * 16 * RT_K + at);
#pragma unroll
      for (int m = 0; m < MT / 2; ++m)
        fx[m] = *reinterpret_cast<const u32x4*>(xl + m * 16 * RT_K + at);
#pragma unroll
      for (int t = 0; t < NT / 2; ++t)
#pragma unroll
        for (int m = 0; m < MT / 2; ++m)
          acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(rg_s16x8, fw[t]),
              __builtin_bit_cast(rg_s16x8, fx[m]), acc[m][t], 0, 0, 0);
    }
  }

  // D[column = lg*4 + r][row = lc] per 16x16 tile
#pragma unroll
  for (int m = 0; m < MT / 2; ++m) {
    const int row = m0 + (wm * MT / 2 + m) * 16 + lc;
    if (row >= M) continue;
    if constexpr (OUT == SILU) {
#pragma unroll
      for (int t = 0; t < NT / 4; ++t) {
        const int col = n0 + wn * 4 * NT + t * 16 + lg * 4;
        if (col >= N) continue;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float g = acc[m][t][j];
          v[j] = g / (1.f + __expf(-g)) * acc[m][t + NT / 4][j];
        }
        uint2 o;
        o.x = (unsigned)f2bf(v[0]) | (unsigned)f2bf(v[1]) << 16;
        o.y = (unsigned)f2bf(v[2]) | (unsigned)f2bf(v[3]) << 16;
        *reinterpret_cast<uint2*>((unsigned short*)out + (long)row * N + col) = o;
      }
      continue;
    }
#pragma unroll
    for (int t = 0; t < NT / 2; ++t) {
      const int col = n0 + (wn * NT / 2 + t) * 16 + lg * 4;
      if (col >= N) continue;               // N is a multiple of 4
      if constexpr (SPLIT) {
        *reinterpret_cast<f32x4*>((float*)out +
                                  ((long)split * M + row) * N + col) = acc[m][t];
      } else {
        uint2 v;
        v.x = (unsigned)f2bf(acc[m][t][0]) | (unsigned)f2bf(acc[m][t][1]) << 16;
        v.y = (unsigned)f2bf(acc[m][t][2]) | (unsigned)f2bf(acc[m][t][3]) << 16;
        *reinterpret_cast<uint2*>((unsigned short*)out + (long)row * N + col) = v;
      }
    }
  }
}

__global__ __launch_bounds__(256) void rows_join_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ parts, long MN,
    int splits) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(parts + i);
  for (int s = 1; s < splits; ++s)
    v += *reinterpret_cast<const f32x4*>(parts + s * MN + i);
  uint2 o;
  o.x = (unsigned)f2bf(v[0]) | (unsigned)f2bf(v[1]) << 16;
  o.y = (unsigned)f2bf(v[2]) | (unsigned)f2bf(v[3]) << 16;
  *reinterpret_cast<uint2*>(out + i) = o;
}

template <int MT, int NT, int S>
void rows_tile(void* out, void* parts, const void* x, const void* w, int M,
               int N, int K, long xs, int splits, bool silu, hipStream_t s) {
  if constexpr (NT >= 4) {
    if (silu) {
      hipLaunchKernelGGL((rows_tile_kernel<MT, NT, S, SILU>),
                         dim3((N + 8 * NT - 1) / (8 * NT)), dim3(256), 0, s, out,
                         (const unsigned short*)x, (const unsigned short*)w, M,
                         N, K, xs, 1);
      return;
    }
  }
  const int nt = (N + 16 * NT - 1) / (16 * NT);
  if (splits > 1 || out == nullptr) {
    hipLaunchKernelGGL((rows_tile_kernel<MT, NT, S, SPLIT_K>),
                       dim3(nt * splits, (M + 16 * MT - 1) / (16 * MT)),
                       dim3(256), 0, s, parts, (const unsigned short*)x,
                       (const unsigned short*)w, M, N, K, xs, splits);
    if (out == nullptr) return;
    const long MN = (long)M * N;
    hipLaunchKernelGGL(rows_join_kernel, dim3((MN / 4 + 255) / 256), dim3(256),
                       0, s, (unsigned short*)out, (const float*)parts, MN,
                       splits);
  } else {
    hipLaunchKernelGGL((rows_tile_kernel<MT, NT, S, ROWS>), dim3(nt),
                       dim3(256), 0, s, out, (const unsigned short*)x,
                       (const unsigned short*)w, M, N, K, xs, 1);
  }
}

template <int NTW>
void rows_gemm(void* out, const void* x, const void* w, int M, int N, int K,
               long xs, hipStream_t s) {
  hipLaunchKernelGGL((rows_gemm_kernel<NTW>),
                     dim3((N + 16 * NTW - 1) / (16 * NTW)), dim3(RG_THREADS),
                     0, s, (unsigned short*)out, (const unsigned short*)x,
                     (const unsigned short*)w, M, N, K, xs);
}

}  // namespace

void rows_gemm_launch(void* out, const void* x, const void* w, int M, int N,
                      int K, long xs, int* err_unsupported, hipStream_t s) {
  *err_unsupported = K % RG_KC != 0 || K == 0 || M > 16;
  if (*err_unsupported || M == 0 || N == 0) return;
  if (N / 32 >= 512) rows_gemm<2>(out, x, w, M, N, K, xs, s);
  else rows_gemm<1>(out, x, w, M, N, K, xs, s);
}

// out [MN] = the sum of the parts [splits, MN], MN a multiple of 4
void rows_join_launch(void* out, const float* parts, long MN, int splits,
                      hipStream_t s) {
  if (MN == 0) return;
  hipLaunchKernelGGL(rows_join_kernel, dim3((MN / 4 + 255) / 256), dim3(256), 0,
                     s, (unsigned short*)out, parts, MN, splits);
}

// parts: fp32 [splits, M, N] where splits > 1, or the result where out is null;
// both for any number of rows. silu: w is [2 N, K], out its activation [M, N].
void rows_tile_launch(void* out, void* parts, const void* x, const void* w,
                      int M, int N, int K, long xs, int cols, int splits,
                      int silu, int* err_unsupported, hipStream_t s) {
  *err_unsupported = K % RT_K != 0 || K == 0 ||
                     (M > 128 && out != nullptr && splits == 1) || N % 4 != 0 ||
                     splits < 1 || splits > K / RT_K ||
                     (cols != 32 && cols != 64 && cols != 128) ||
                     (silu && (splits != 1 || cols == 32 || out == nullptr));
  if (*err_unsupported || M == 0 || N == 0) return;
  const int wide = silu ? 2 * N : N;
#define RT(MT, S2, S4, S8)                                                    \
  if (cols == 32) rows_tile<MT, 2, S2>(out, parts, x, w, M, N, K, xs, splits, silu, s); \
  else if (cols == 64) rows_tile<MT, 4, S4>(out, parts, x, w, M, N, K, xs, splits, silu, s); \
  else rows_tile<MT, 8, S8>(out, parts, x, w, M, N, K, xs, splits, silu, s);
  if (M <= 32) { RT(2, 8, 6, 4) }
  else if (M <= 64) { RT(4, 6, 5, 3) }
  else if ((wide + cols - 1) / cols * splits * ((M + 127) / 128) <= 256) {
    // one workgroup a CU
    if (M <= 96) { RT(6, 8, 7, 5) }
    else { RT(8, 7, 6, 4) }
  }
  else if (M <= 96) { RT(6, 5, 4, 2) }
  else { RT(8, 4, 3, 2) }
#undef RT
}
