// Products with packed int4 weights for MI355X (gfx950): out[M, N] =
// x[M, K] W^T with W kept packed in HBM, and the transient expansion to bf16
// that prompt-sized products use in front of the library GEMM.
//
// Packed layout (models/quantized.py pack_w4_runtime): qw u8 [N, K/2] in
// FRAGMENT ORDER: within each 128-k block, the 16 bytes that lane group lg loads
// hold the 32 weights (4 MFMA k-chunks x 8 values) of its operand fragments, word
// c those of k = c*32 + lg*8 .. + 7. In a word value j is the nibble at bit
// 4*(j/2) + 16*(j%2): neighbours lie 16 bits apart, as in a register of bf16.
// Scales / zero-scales: bf16 [N, K/128], one group per 128-k block.
// w = q * s - zs   (zs = zero * s, precomputed).
//
// A nibble becomes bf16 without arithmetic: 0x4300 | q is 128 + q, two at a time.
// The products of a block are exact in q; its scale and offset are applied to the
// fp32 sums:
//   out += s * (x . (128 + q)) - (128 s + zs) * sum(x),
// sum(x) coming from a product with a fragment of ones. The weights are never
// rounded to bf16 here, as the expansion does.
//
// Tiles (w4_tile_kernel). 8 waves (4 where the columns are no multiple of 128)
// have 16 columns each and all of up to 64 rows; more rows are more workgroups.
// Steps of 256 k of x and of the weights go to two buffers in the LDS, whole
// 128-byte lines of both by loads that write the LDS themselves, one step ahead; or 16
// waves, two to a column tile with half a step each, whose sums meet at the end.
// 16-byte chunks are permuted through the lanes' addresses: of x's rows (512
// bytes) XORed with the row, of the weights' (128 bytes) with (row >> 1). Weights
// are the A operand: a lane ends with 4 neighbouring columns of a row. The sums of
// x over a step's blocks are made once, by a wave each, and used a step later.
// Narrow products are cut over k into fp32 parts, which the next kernel adds up.
// What bounds it is a wave's chain in a step, LDS, unpacking, products and scales, of
// which four waves a SIMD hide more than two; at 64 rows the reads of x from the LDS. us,
// weights out of memory, 8 waves with scales one by one -> now at 8 / 16 / 32 / 64 rows:
// 28672 x 4096 with the activation 21.3 -> 17.2 / 22.2 -> 18.3 / 23.7 -> 21.2 / 32.9 ->
// 27.3, 57344 x 8192 59 -> 55 / 67 -> 59 / 87 -> 78 / 120 -> 100, 128256 x 4096 61 -> 57
// / 61 -> 58 / 95 -> 83 / 128 -> 107, 8192 x 28672 28 -> 28.6 / 29.7 -> 29.0 / 43 -> 37.5
// / 57 -> 49, 4096 x 14336 11.7 -> 10.9 / 11.8 -> 11.2 / 13.0 -> 13.1 / 17.6 -> 17.0.
// A step's addresses are a number the wave shares and 32 bits of offset a lane, and its
// buffer is a constant of the code (64-bit addresses of each lane, made anew in every
// step -> this, at 16 / 32 / 64 / 100 rows: 57344 x 8192 62 -> 57 / 84 -> 82 / 106 -> 103
// / 208 -> 191, 128256 x 4096 63 -> 60 / 88.7 -> 89 / 114 -> 110 / 221 -> 211, 4096 x
// 14336 12.4 -> 12.1 / 14.1 -> 14.2 / 17.6 -> 17.3 / 32 -> 30.6, in four waves 5184 x
// 8192 10.9 / 16.3 -> 15.1 / 22.9 -> 20.9 / 42.5 -> 38.3).
// Two tiles of columns a wave, four waves: 27, 14, 9.1, 6.2, 73 at 16 rows and 42,
// 22, 15, 9.9, 173 at 64 (28672 x 4096, 4096 x 14336, 6144 x, 4096 x, 128256 x 4096).
//
// Rows (w4_rows_kernel): few rows of products that are narrow and have no consumer
// for parts, and small ones. Straight from memory, k cut over the waves.
#include "common.h"

#include <type_traits>

namespace {

constexpr int W4_KC = 128;

typedef __attribute__((ext_vector_type(8))) short w4_s16x8;

DEVICE_INLINE f32x4 w4_mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(w4_s16x8, a), __builtin_bit_cast(w4_s16x8, b), c, 0, 0, 0);
}

// eight nibbles as bf16 128 + q, in order. FUSED: the mask in a scalar and the exponents
// in a vector register, both hidden from the compiler, which else takes two instructions
// for the v_and_or_b32 that has no room for two constants (with 16 waves 3 to 8 %; where
// a workgroup has 8, waves wait for the memory, and 128256 columns took 65 us for 61).
template <bool FUSED = false>
DEVICE_INLINE u32x4 w4_bf16(unsigned int d) {
  unsigned int mask = 0x000f000fu, high = 0x43004300u;
  if constexpr (FUSED) {
    asm("" : "+s"(mask));
    asm("" : "+v"(high));
  }
  u32x4 o;
#pragma unroll
  for (int j = 0; j < 4; ++j) o[j] = ((d >> (4 * j)) & mask) | high;
  return o;
}

constexpr int W4_SK = 2 * W4_KC;            // k of a step
constexpr int W4_SZ = 32;                   // blocks of k whose scales are staged

// What becomes of the sums: the result, fp32 parts [splits, M, N], or
// silu(gate) * up in [M, N], qw then holding N gate rows and N up rows behind.
enum W4Out { W4_ROWS, W4_PARTS, W4_SILU };

// KW 2: twice the waves, each with one of a step's two blocks. NB: buffers in the LDS.
template <int MT, int WAVES, int KW, int NB, W4Out OUT>
__global__ __launch_bounds__(WAVES * KW * WAVE_SIZE) void w4_tile_kernel(
    void* __restrict__ out, const unsigned short* __restrict__ x,  // [M, K] bf16
    const unsigned char* __restrict__ qw,   // [N, K/2] frag-ordered nibbles
    const unsigned short* __restrict__ sc,  // [N, K/128] bf16 scale
    const unsigned short* __restrict__ zs,  // [N, K/128] bf16 zero*scale
    int M, int N, int K, int splits) {
  constexpr int ROWS = 16 * MT, COLS = 16 * WAVES;
  constexpr int XB = ROWS * W4_SK, BUF = XB + COLS * 64;  // elements of 2 bytes
  constexpr int ALL = WAVES * KW;
  constexpr int LX = (8 * MT + ALL - 1) / ALL;  // loads of x of a wave in a step
  constexpr int LW = 2 / KW;                // of its weights
  constexpr int CT = OUT == W4_SILU ? COLS / 2 : COLS;    // columns of out
  __shared__ __attribute__((aligned(1024))) unsigned short lds[NB * BUF];
  __shared__ __attribute__((aligned(16))) unsigned int sz[W4_SZ * COLS];
  __shared__ float xsum[2][2][ROWS];        // of a step's blocks, by its parity

  const int nb = K / W4_KC, total = (nb + 1) / 2;
  const bool pairs = nb % 2 == 0 && ((unsigned long)sc | (unsigned long)zs) % 4 == 0;
  const int split = OUT == W4_PARTS ? blockIdx.x % splits : 0;
  const int n0 = (OUT == W4_PARTS ? blockIdx.x / splits : blockIdx.x) * CT;
  const int m0 = blockIdx.y * ROWS;
  int from = 0, end = total;
  if constexpr (OUT == W4_PARTS) {
    from = (int)((long)total * split / splits);
    end = (int)((long)total * (split + 1) / splits);
  }
  const int tid = threadIdx.x, lane = tid & (WAVE_SIZE - 1);
  const int any = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wave = any % WAVES, kw = any / WAVES;  // columns, and half of a step
  const int lc = lane & 15, lg = lane >> 4;
  // row of qw of one of the workgroup's columns: the first waves' are of the gate
  auto at = [&](int c) {
    return n0 + c + (OUT == W4_SILU && c >= CT ? N - CT : 0);
  };

  // an instruction brings 2 rows of x, or 8 of the weights, a wave its own
  // columns; a step of one block (the last of an odd number) brings it twice. Lanes keep
  // offsets, what changes from step to step is the wave's.
  unsigned int xo[LX], wo[LW];
  int xc[LX], wc[LW];
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (any * LX + i) * 2 + lane / 32;
    xc[i] = (lane & 31) ^ (row & 15);
    xo[i] = ((unsigned)min(row, M - 1 - m0) * (unsigned)K + xc[i] * 8) * 2;
  }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (kw * LW + i) * 8 + lane / 8;
    wc[i] = (lane & 7) ^ ((row >> 1) & 7);
    wo[i] = (unsigned)row * (unsigned)(K / 2) + wc[i] * 16;
  }
  const unsigned char* wbase = qw + (long)at(wave * 16) * (K / 2);

  f32x4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
  constexpr int HB = 2 / KW;                // blocks of a step that are the wave's
  f32x4 z[HB];                              // 128 s + zs of the step before
  auto correct = [&](int i) {
#pragma unroll
    for (int h = 0; h < HB; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float xs = xsum[i & 1][kw * HB + h][m * 16 + lc];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] -= z[h][r] * xs;
      }
  };

  for (; from < end; from += W4_SZ / 2) {    // once up to 4096 k
    const int n = min(end - from, W4_SZ / 2);
    // Steps start at the workgroup's own place in the row: rows lie a power of
    // two apart, and workgroups that all read the same columns of their rows
    // would meet on a few memory channels.
    const int rot = blockIdx.x % n;
    auto step = [&](int i) {
      return from + (i + rot < n ? i + rot : i + rot - n);
    };
    auto stage = [&](int i, int in) {
      const int st = step(i);
      const bool half = 2 * st + 1 >= nb;
      unsigned short* to = lds + in * BUF;
      const unsigned short* xb = x + (long)m0 * K + (long)st * W4_SK;
      const unsigned short* wb =
          reinterpret_cast<const unsigned short*>(wbase + (long)st * W4_KC);
      auto bring = [&](auto twice) {
#pragma unroll
        for (int j = 0; j < LX; ++j)
          if (8 * MT >= ALL || any * LX + j < 8 * MT)
            load_to_lds(xb, twice.value ? xo[j] - (xc[j] & 16) * 16 : xo[j],
                        to + (any * LX + j) * 2 * W4_SK);
#pragma unroll
        for (int j = 0; j < LW; ++j)
          load_to_lds(wb, twice.value ? wo[j] - (wc[j] & 4) * 16 : wo[j],
                      to + XB + (wave * 16 + (kw * LW + j) * 8) * 64);
      };
      if (half) bring(std::true_type{});
      else bring(std::false_type{});
    };
    for (int i = 0; i < NB - 1 && i < n; ++i) stage(i, i);
    // scale (low half) and offset of every column and block, 0 behind the last; two
    // blocks at a time where they lie so (28672 x 4096 22 -> 20 us)
    const int b0 = 2 * from;
    if (pairs) {
#pragma unroll 4
      for (int u = tid; u < COLS * n; u += ALL * WAVE_SIZE) {
        const int c = u / n, b = u % n;
        const long i = ((long)at(c) * nb + b0) / 2 + b;
        const unsigned int p = reinterpret_cast<const unsigned int*>(sc)[i];
        const unsigned int q = reinterpret_cast<const unsigned int*>(zs)[i];
        sz[2 * b * COLS + c] = (p & 0xffffu) | (q << 16);
        sz[(2 * b + 1) * COLS + c] = (p >> 16) | (q & 0xffff0000u);
      }
    } else {
      for (int u = tid; u < COLS * 2 * n; u += ALL * WAVE_SIZE) {
        const int c = u / (2 * n), b = u % (2 * n);
        const long i = (long)at(c) * nb + b0 + b;
        sz[b * COLS + c] =
            b0 + b < nb ? (unsigned int)sc[i] | ((unsigned int)zs[i] << 16) : 0u;
      }
    }

    // step i, in a buffer of the LDS whose number is a constant of the code
    auto work = [&](int i, auto in) {
      constexpr int B = decltype(in)::value;
      // the steps asked for behind this one; a wave may have no rows of x to bring
      if (NB > 2 && i > 0 && i + NB - 2 < n)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)"
                     ::"n"((NB - 2) * (8 * MT >= ALL ? LX + LW : LW)) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (i + NB - 1 < n) stage(i + NB - 1, (B + NB - 1) % NB);
      if (i > 0) correct(i - 1);
      const unsigned short* xl = lds + B * BUF + lc * W4_SK;
      const unsigned short* wl =
          lds + B * BUF + XB + (wave * 16 + lc) * 64;
      const int b = 2 * (step(i) - from);
      // sums of x over the blocks, each by one of the waves for all
#pragma unroll
      for (int j = 0; j < (2 * MT + ALL - 1) / ALL; ++j) {
        const int q = any + j * ALL, h = q / MT, m = q % MT;
        if (q >= 2 * MT) break;
        f32x4 xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c)
          xs = w4_mfma(ones,
                       *reinterpret_cast<const u32x4*>(
                           xl + m * 16 * W4_SK + ((h * 16 + c * 4 + lg) ^ lc) * 8),
                       xs);
        if (lg == 0) xsum[i & 1][h][m * 16 + lc] = xs[0];
      }
#pragma unroll
      for (int hh = 0; hh < HB; ++hh) {
        const int h = kw * HB + hh;
        const u32x4 w4 = *reinterpret_cast<const u32x4*>(
            wl + ((h * 4 + lg) ^ ((lc >> 1) & 7)) * 8);
        f32x4 p[MT];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const u32x4 wf = w4_bf16<KW == 2>(w4[c]);
#pragma unroll
          for (int m = 0; m < MT; ++m)
            p[m] = w4_mfma(wf,
                           *reinterpret_cast<const u32x4*>(
                               xl + m * 16 * W4_SK +
                               ((h * 16 + c * 4 + lg) ^ lc) * 8),
                           c ? p[m] : f32x4{0.f, 0.f, 0.f, 0.f});
        }
        const u32x4 v = *reinterpret_cast<const u32x4*>(
            sz + (b + h) * COLS + wave * 16 + lg * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float s = __builtin_bit_cast(float, v[r] << 16);
          z[hh][r] = 128.f * s + __builtin_bit_cast(float, v[r] & 0xffff0000u);
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][r] += s * p[m][r];
        }
      }
    };
    for (int i = 0; i < n; i += NB) {
      work(i, std::integral_constant<int, 0>{});
      if (i + 1 < n) work(i + 1, std::integral_constant<int, 1>{});
      if constexpr (NB > 2) {
        if (i + 2 < n) work(i + 2, std::integral_constant<int, 2>{});
        if (i + 3 < n) work(i + 3, std::integral_constant<int, 3>{});
      }
    }
    __syncthreads();
    correct(n - 1);
    __syncthreads();                         // the buffers are done with
  }

  // the halves of the steps together
  if constexpr (KW == 2) {
    f32x4* other = reinterpret_cast<f32x4*>(lds) + wave * MT * WAVE_SIZE + lane;
    if (kw == 1)
#pragma unroll
      for (int m = 0; m < MT; ++m) other[m * WAVE_SIZE] = acc[m];
    __syncthreads();
    if (kw == 0)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const f32x4 v = other[m * WAVE_SIZE];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] += v[r];
      }
    __syncthreads();
  }

  // D[column = lg*4 + r][row = lc]
  constexpr int US = CT + 4;                 // the up product's rows in the LDS
  float* up = reinterpret_cast<float*>(lds);
  if constexpr (OUT == W4_SILU) {
    if (wave >= WAVES / 2 && kw == 0)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        *reinterpret_cast<f32x4*>(up + (m * 16 + lc) * US +
                                  (wave - WAVES / 2) * 16 + lg * 4) = acc[m];
    __syncthreads();
    if (wave >= WAVES / 2) return;
  }
  if (kw > 0) return;
  const int col = n0 + wave * 16 + lg * 4;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m0 + m * 16 + lc;
    if (row >= M) continue;
    f32x4 v = acc[m];
    if constexpr (OUT == W4_PARTS) {
      *reinterpret_cast<f32x4*>((float*)out + ((long)split * M + row) * N + col) =
          v;
    } else {
      if constexpr (OUT == W4_SILU) {
        const f32x4 u = *reinterpret_cast<const f32x4*>(
            up + (m * 16 + lc) * US + wave * 16 + lg * 4);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = v[r] / (1.f + __expf(-v[r])) * u[r];
      }
      uint2 o;
      o.x = (unsigned)f2bf(v[0]) | (unsigned)f2bf(v[1]) << 16;
      o.y = (unsigned)f2bf(v[2]) | (unsigned)f2bf(v[3]) << 16;
      *reinterpret_cast<uint2*>((unsigned short*)out + (long)row * N + col) = o;
    }
  }
}

template <int NTW, int WAVES>
__global__ __launch_bounds__(WAVES * WAVE_SIZE) void w4_rows_kernel(
    unsigned short* __restrict__ out,       // [M, N] bf16
    const unsigned short* __restrict__ x,   // [M, K] bf16
    const unsigned char* __restrict__ qw,   // [N, K/2] frag-ordered nibbles
    const unsigned short* __restrict__ sc,  // [N, K/128] bf16 scale
    const unsigned short* __restrict__ zs,  // [N, K/128] bf16 zero*scale
    int M, int N, int K) {
  constexpr int COLS = 16 * NTW, ROWS = 16;
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
  const unsigned short* xp = x + (long)min(m0 + lc, M - 1) * K + lg * 8;

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

  f32x4 acc[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};

  auto multiply = [&](int b) {
    u32x4 xa[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      xa[c] = *reinterpret_cast<const u32x4*>(xp + b * W4_KC + c * 32);
    f32x4 xs = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c) xs = w4_mfma(xa[c], ones, xs);
#pragma unroll
    for (int t = 0; t < NTW; ++t) {
      f32x4 p = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) p = w4_mfma(xa[c], w4_bf16(wc[t][c]), p);
      const unsigned int v = sz[b * COLS + t * 16 + lc];
      const float s = __builtin_bit_cast(float, v << 16);
      const float z = 128.f * s + __builtin_bit_cast(float, v & 0xffff0000u);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[t][r] += s * p[r] - z * xs[r];
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
  for (int t = 0; t < NTW; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      red[(wave * ROWS + lg * 4 + r) * COLS + t * 16 + lc] = acc[t][r];
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
        o[j] = f2bf((float)((d >> (j / 2 * 4 + j % 2 * 16)) & 0xF) * s - z);
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
template <int NTW, int WAVES>
void w4_rows(void* out, const void* x, const void* qw, const void* sc,
             const void* zs, int M, int N, int K, hipStream_t s) {
  const size_t scales = (size_t)(K / W4_KC) * 16 * NTW * 4;
  const size_t sums = (size_t)WAVES * 16 * 16 * NTW * 4;
  hipLaunchKernelGGL((w4_rows_kernel<NTW, WAVES>),
                     dim3(N / (16 * NTW), (M + 15) / 16),
                     dim3(WAVES * WAVE_SIZE), scales > sums ? scales : sums, s,
                     (unsigned short*)out, (const unsigned short*)x,
                     (const unsigned char*)qw, (const unsigned short*)sc,
                     (const unsigned short*)zs, M, N, K);
}

template <int MT, int WAVES, int KW, int NB, W4Out OUT>
void w4_tile(void* out, const void* x, const void* qw, const void* sc,
             const void* zs, int M, int N, int K, int splits, hipStream_t s) {
  constexpr int CT = (OUT == W4_SILU ? 8 : 16) * WAVES;
  hipLaunchKernelGGL((w4_tile_kernel<MT, WAVES, KW, NB, OUT>),
                     dim3(N / CT * splits, (M + 16 * MT - 1) / (16 * MT)),
                     dim3(WAVES * KW * WAVE_SIZE), 0, s, out,
                     (const unsigned short*)x, (const unsigned char*)qw,
                     (const unsigned short*)sc, (const unsigned short*)zs, M, N,
                     K, splits);
}

int w4_waves(int N) { return N % 128 == 0 ? 8 : 4; }

template <W4Out OUT>
void w4_tiles(void* out, const void* x, const void* qw, const void* sc,
              const void* zs, int M, int N, int K, int splits, hipStream_t s) {
  // Sixteen waves for eight from four steps a workgroup on (us, eight / sixteen, 16 rows
  // and 64: 28672 x 4096 20.2 / 20.3 and 30.7 / 27.3, 57344 x 8192 63 / 59 and 113 / 100,
  // 128256 x 4096 65 / 58 and 123 / 107; but 4096 x 4096, two steps, 5.7 / 5.9), with two
  // more buffers where every workgroup has a CU of its own (28672 x 4096 20.3 / 18.3, at
  // 57344 x 8192 59 / 66).
  const int groups = (OUT == W4_SILU ? N / 64 : N / (16 * w4_waves(N))) * splits;
  const bool half = (K / W4_KC + 1) / 2 / splits >= 4, own = groups <= 256;
#define W4_TILE(MT)                                                                \
  do {                                                                             \
    if (OUT != W4_SILU && w4_waves(N) == 4) {                                      \
      if constexpr (OUT != W4_SILU)                                                \
        w4_tile<MT, 4, 1, 2, OUT>(out, x, qw, sc, zs, M, N, K, splits, s);         \
    } else if (!half) {                                                            \
      w4_tile<MT, 8, 1, 2, OUT>(out, x, qw, sc, zs, M, N, K, splits, s);           \
    } else if (MT == 1 && own) {                                                   \
      w4_tile<MT, 8, 2, MT == 1 ? 4 : 2, OUT>(out, x, qw, sc, zs, M, N, K, splits, s); \
    } else {                                                                       \
      w4_tile<MT, 8, 2, 2, OUT>(out, x, qw, sc, zs, M, N, K, splits, s);           \
    }                                                                              \
  } while (0)
  if (M <= 16) W4_TILE(1);
  else if (M <= 32) W4_TILE(2);
  else W4_TILE(4);
#undef W4_TILE
}
}  // namespace

// Shapes that have a product: whole workgroups of 64 columns, blocks of 128 k.
bool w4_has(int N, int K) {
  return N % 64 == 0 && K % W4_KC == 0 && K > 0 && K / W4_KC <= 1024;
}

// Parts over k: one workgroup a CU, up to 16 rows of long rows two, 8 parts at
// most. us at 16 rows in 8 waves: 4096 x 14336 (32 groups) 4 parts 20, 8 12, 16 13;
// 6144 x 4096 (48) 2 12, 5 7.4, 8 7.3; 8192 x 28672 (64) 4 37, 8 29; 10240 x 8192 (80)
// 3 16, 6 15; at 64 rows: 6144 x 4096 5 12, 8 15; 10240 x 8192 3 25, 6 30. In 16 waves
// those taken are 12.0, 7.8, 30.7, 16.6, 12.4 and 23.0.
int w4_splits(int M, int N, int K) {
  const int groups = N / (16 * w4_waves(N)), total = (K / W4_KC + 1) / 2;
  int splits = (M <= 16 && K >= 8192 ? 512 : 256) / groups;
  if (splits > 8) splits = 8;
  if (splits > total) splits = total;
  return splits > 1 ? splits : 1;
}

// Products for which parts do not pay even where the next kernel adds them up: few
// rows of short ones (at one row, with a norm behind, 6144 x 4096 10.0 against 12.3 and
// 4096 x 4096 7.8 against 10.1, but 8192 x 28672 43 / 36), and small ones (6144 x 1920
// at 16 rows 5.0 / 5.3). Of 640 sizes 81 of those that are cut take more than 3 % longer
// than whole, to 1.28 (one row of 4096 x 8192 10.9 / 14.0), 44 of the others would gain
// that (48 rows of 3072 x 4096 19 / 14).
bool w4_cuts(int M, int N, int K) {
  return (M >= 8 || K >= 8192) && (long)N * K > 12l << 20 &&
         w4_splits(M, N, K) > 1;
}

// The whole result: rows where these are few and the product is narrow, as far as a
// wave of the rows' form has two column tiles (w4_rows_launch; us against the tiles, 24576
// x 4096 at one row 16.5 / 17.4, at 8 18.4 / 17.2; with four tiles 28672 x 4096 21.1 /
// 17.7 and 22.1 / 18.0), unless k is long and parts with a join (3 us) gain more (4096
// x 14336 at 16 rows 20 against 12 + 3), and for small products (6144 x 1920 at 64 rows
// 10 against 8 + 3). Left on the wrong side: more than 8 rows of 12288 columns and more
// that do not end in the activation (24576 x 4096 at 16 rows 22.4 / 17.6), 10240 columns
// and more of 8192 k and more at any (8 rows of 10240 x 14336 38 / 25).
bool w4_by_rows(int M, int N, int K) {
  if (M <= 16 && N < 28672 && !(M > 8 && K >= 8192)) return true;
  return M <= 64 && (long)N * K <= 12l << 20;
}

// Whether a product of N columns (gate and up) ends in the activation. Where the
// product is one launch of whole tiles by itself it does, and saves the
// activation's launch (us without / with, 28672 x 4096 at 16 rows 20.6 / 18.2, 24 rows
// 24.4 / 21.9, 64 rows 31.5 / 28.0, 192 rows 85 / 80; 17920 x 2048 at 64 rows 18.7 /
// 15.7). Products cut over k do not: their chain of k would run whole on less than one
// workgroup a CU (16384 x 4096 at 64 rows 25 / 27; 22016 x 8192 at 16 rows, right on
// it, 33.9 / 33.5).
// In the place of the rows' form, up to 16 rows, the tiles pay for a chain of .8
// microseconds for every 256 k, however few rows there are, and the rows' form for
// its columns and for x, which it reads again in every workgroup: the line grows
// with both (22016 columns at one row x 2048 12.4 / 10.7, x 4096 18.2 / 17.0, x 5120,
// right on it, 21.5 / 22.3, x 8192 31.2 / 33.0; 17920 x 5120 at 2 rows 21.0 / 21.6, at 8
// rows 23.9 / 21.6). It lies where the tiles take .8 us more in these loops: in a captured step
// the activation costs 1.5 us more besides.
bool w4_silu_wins(int M, int N, int K) {
  if (w4_by_rows(M, N, K))
    return M <= 16 && N > 16384 && K < 256 * (M + 16) + (N - 16384) / 4;
  return w4_splits(M, N, K) == 1;
}

// parts: fp32 [splits, M, N]. x, qw and parts at 16-byte addresses.
void w4_parts_launch(float* parts, const void* x, const void* qw, const void* sc,
                     const void* zs, int M, int N, int K, int splits,
                     hipStream_t s) {
  if (M > 0) w4_tiles<W4_PARTS>(parts, x, qw, sc, zs, M, N, K, splits, s);
}

// out [M, N] = silu(gate) * up, qw of N gate rows and N up rows, N a multiple of
// 64. x, qw and out at 16-byte addresses.
void w4_silu_launch(void* out, const void* x, const void* qw, const void* sc,
                    const void* zs, int M, int N, int K, hipStream_t s) {
  if (M > 0) w4_tiles<W4_SILU>(out, x, qw, sc, zs, M, N, K, 1, s);
}

// One launch. x, qw and out at 16-byte addresses.
void w4_tile_launch(void* out, const void* x, const void* qw, const void* sc,
                    const void* zs, int M, int N, int K, hipStream_t s) {
  if (M > 0) w4_tiles<W4_ROWS>(out, x, qw, sc, zs, M, N, K, 1, s);
}

// The form by columns: workgroups of four column tiles per wave from 448 of them
// on; of two from 160 on, with 16 waves (6144 x 4096, us at 16 rows: 9.1 against
// 12.3 with one tile); else of one, which keeps every CU on the stream (4096 x
// 4096 at 16 rows: 7.6 against 8.7 with two), with 16 waves for long rows (4096 x
// 14336 at one row: 11.9 against 14.5). The scales of K / 128 blocks stay under
// 64 KB.
void w4_rows_launch(void* out, const void* x, const void* qw, const void* sc,
                    const void* zs, int M, int N, int K, hipStream_t s) {
  if (M == 0) return;
  const int nb = K / W4_KC;
  const int ntw = N / 64 >= 448 && nb <= 256 ? 4
                  : N / 32 >= 160 && nb <= 512 ? 2 : 1;
#define W4_ARGS out, x, qw, sc, zs, M, N, K, s
  if (ntw == 4) w4_rows<4, 8>(W4_ARGS);
  else if (ntw == 2) w4_rows<2, 16>(W4_ARGS);
  else if (nb >= 64) w4_rows<1, 16>(W4_ARGS);
  else w4_rows<1, 8>(W4_ARGS);
#undef W4_ARGS
}
