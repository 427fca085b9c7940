// Products of many rows for MI355X (gfx950) in tiles of 256 rows and 256 weight
// rows: silu(x Wg^T) * (x Wu^T) in one launch, or x W^T cut over k.
//
// One workgroup a CU walks its tiles; four waves of 128 x 128 on
// mfma_f32_16x16x32_bf16 (of random numbers 2.1 PFLOP/s before the card's power
// limits it, 32x32x16 1.85), fp32 sums in the accumulation registers. Larger waves
// read less: 64 x 64 ask the LDS for 128 bytes a cycle at the full matrix rate, which
// is all that it has, these for 64, and the L1 for 32 where tiles of 128 x 128 ask it
// for the 64 that it has.
// A step is 64 k: rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 % 8), which
// 16 rows of one chunk read without conflict. (Rows of 32 k, five steps deep: 1530 us
// where these take 1390, 8192 rows of 28672 x 4096; the L1 serves half lines.) Two
// buffers of rows and three of weights fill the LDS; buffers of a step are asked for
// two steps ahead, through the end of a tile into the next one, whose first steps come
// while the results of this one are stored.
// With one wave a SIMD the matrix unit idles whenever the wave issues more than two or
// three other instructions between two products: operands are read half a step ahead,
// and each gap between products holds one LDS read or one load, no branch (8 loads
// behind every eighth product 1390 us, one in every eighth gap 1310).
// The products are inline asm that adds in place: left to itself the compiler writes
// them to other registers and copies, all 256 being taken. It does not see the products
// in the asm, so the waits before their results are read stand here (s_nop), and a loop
// of one body keeps it from copying them in between.
// 8192 rows of 28672 x 4096 with the activation 1228 us (1566 TFLOP/s), 2039 rows 345
// (3.5 rounds of tiles in the time of four), 512 rows 86 (1403), 91 out of HBM; the
// library's product and the activation behind it 1290 + 127, 353 + 31, 85 + 11.
// A product of fewer columns leaves workgroups without a tile: cut over k it fills them,
// and what reads it adds the fp32 parts up: with an RMS norm behind, 4096 x 14336 at 512
// rows 69 us (before 73), 640 84 (143), 1024 107 (159), 2039 197 (217).
// Without the activation and whole, the tiles are 1.00 to 1.05 of the library's time.
#include "wide_tiles.h"

namespace {

constexpr int WT_ROWS = 256, WT_K = 64;
constexpr int WT_BUF = WT_ROWS * WT_K;      // elements of a buffer
constexpr int WT_BYTES = WT_BUF * 2;
constexpr int WT_CUS = 256;                 // workgroups of a launch

// SILU: out [M, N] = silu(x Wg^T) * (x Wu^T), w [2 N, K] = Wg, then Wu. PARTS: out
// [splits, M, N] = x W^T in fp32, each of its own steps of k, w [N, K].
enum WideOut { SILU, PARTS };

template <int OUT>
__global__ __launch_bounds__(256, 1) void wide_kernel(
    void* __restrict__ out_, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, int M, int N, int K, long xs, int splits) {
  constexpr int COLS = OUT == SILU ? WT_ROWS / 2 : WT_ROWS;  // columns of a tile
  constexpr int HC = COLS / 2;              // of a wave
  // of a wave at the end of a tile; what a wait can count
  constexpr int STORES = OUT == SILU ? 16 : 55;
  // rows' buffers, then the weights'
  __shared__ __attribute__((aligned(16))) unsigned short lds[5 * WT_BUF];
  const int tid = threadIdx.x, lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave >> 1, wn = wave & 1;
  const int lc = lane & 15, lg = lane >> 4;
  const int steps = K / WT_K;
  const int WN = OUT == SILU ? 2 * N : N;   // weight rows
  const int mt = (M + WT_ROWS - 1) / WT_ROWS, nt = (N + COLS - 1) / COLS;

  // An XCD's tiles follow each other in blocks of 8 tiles of rows by all columns,
  // rows first, so that its L2 serves 8 workgroups a weight and 4 a row; one part of
  // k behind the other.
  const int xcd = blockIdx.x & 7, per = WT_CUS / 8, slot = blockIdx.x >> 3;
  const int all = mt * nt * (OUT == PARTS ? splits : 1);
  const int q = all / 8, r = all % 8;
  const int count = xcd < r ? q + 1 : q;    // tiles of this XCD
  const int start = xcd * q + min(xcd, r);
  if (slot >= count) return;
  const int rounds = (count - slot + per - 1) / per;
  struct Place { int m0, n0, part, from, n; };  // n: steps, the first is `from`
  auto one = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  auto place = [&](int round) {
    int t = start + round * per + slot;
    Place p{0, 0, 0, 0, steps};
    if constexpr (OUT == PARTS) {
      p.part = t / (mt * nt);
      t -= p.part * (mt * nt);
      p.from = one((int)((long)steps * p.part / splits));
      p.n = one((int)((long)steps * (p.part + 1) / splits)) - p.from;
    }
    const int g = t / (8 * nt), in = t % (8 * nt), high = min(8, mt - g * 8);
    p.m0 = one((g * 8 + in % high) * WT_ROWS);
    p.n0 = one(in / high * COLS);
    return p;
  };

  // A wave's load i brings rows (i * 4 + wave) * 8 .. of 128 bytes to the LDS. Row
  // 4 g + j of a wave's tiles 2 p and 2 p + 1 is column 32 p + 8 g + j and + 4, so that
  // a lane ends with eight neighbouring columns; of SILU tiles 0 to 3 are the gate's, 4
  // to 7 the up product's.
  unsigned ox[8], ow[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    const int at = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    const int b = (row >> 4) & (OUT == SILU ? 3 : 7), ii = row & 15;
    const int col = (row >> 7) * HC + (b >> 1) * 32 + (ii >> 2) * 8 + (b & 1) * 4 +
                    (ii & 3) + (OUT == SILU && (row & 64) ? N : 0);
    ox[i] = ((unsigned)row * (unsigned)xs + at) * 2;
    ow[i] = ((unsigned)col * (unsigned)K + at) * 2;
  }
  const int at0 = lc * WT_K + (lg ^ ((lc >> 1) & 7)) * 8, at1 = at0 ^ 32;
  const unsigned short* wl = lds + (2 * WT_ROWS + wn * 128) * WT_K;
  const unsigned to = lds_address(lds) + wave * 8 * WT_K * 2;

  // The step that is loaded next: of the tile of round `lr`, with `left` steps to come;
  // k0: its bytes from the start of a row. Weight rows lie a power of two apart, and
  // workgroups at one place of theirs meet on a few memory channels: each XCD begins an
  // eighth of the row further on (512 rows of 28672 x 4096 out of HBM 97 -> 91 us; each
  // column tile at a place of its own 96, and 1327 for 1250 at 8192 rows, whose rows
  // then miss the L2). Of no use in more rows, which compute longer than they load
  // (7122 x 8192 x 2048 330 -> 331), and parts begin elsewhere anyway.
  const int turn = OUT == SILU && M <= 2048 ? xcd * steps / 8 : 0;
  int lr = 0, left = 0;
  unsigned k0 = 0;
  i32x4 rx{}, rw{};
  auto point = [&]() {
    if (lr < rounds) {
      const Place p = place(lr);
      left = p.n;
      k0 = (unsigned)(OUT == PARTS ? p.from : turn) * (WT_K * 2);
      rx = wt_rsrc(x + p.m0 * xs, ((unsigned)min(WT_ROWS, M - p.m0) - 1) *
                                          (unsigned)xs * 2 + (unsigned)K * 2);
      rw = wt_rsrc(w + (long)p.n0 * K, (unsigned)(WN - p.n0) * (unsigned)K * 2);
    } else {
      left = steps;
      k0 = 0;
      rx[2] = rw[2] = 0;
    }
  };
  auto advance = [&]() {
    k0 += WT_K * 2;
    if (OUT == SILU && k0 == (unsigned)K * 2) k0 = 0;
    if (--left == 0) {
      ++lr;
      point();
    }
  };
  auto load = [&](unsigned at, unsigned off, const i32x4& rs) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(at), "v"(off), "s"(rs), "s"(k0)
                 : "m0", "memory");
  };
  point();
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      load(to + (2 + s) * WT_BYTES + i * 4096, ow[i], rw);
#pragma unroll
    for (int i = 0; i < 8; ++i) load(to + s * WT_BYTES + i * 4096, ox[i], rx);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int bx = 0, bw = 0;                       // buffers of the step at hand

  const unsigned short* rl = lds + wm * 128 * WT_K;
  u32x4 fr[2][8], fw[2][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    fw[0][i] = *reinterpret_cast<const u32x4*>(wl + at0 + i * 16 * WT_K);
    fr[0][i] = *reinterpret_cast<const u32x4*>(rl + at0 + i * 16 * WT_K);
  }
  f32x4 acc[8][8];

  // The products of half `h` of a step; into the gaps between them go the operands of
  // the next half, from rn and wnx, and eight loads to `dst`.
  auto half = [&](auto h, const unsigned short* rn, const unsigned short* wnx,
                  const i32x4& rs, unsigned dst, const unsigned* off) {
    constexpr int H = decltype(h)::value;
#pragma unroll
    for (int i = 0; i < 64; ++i) {
      const int a = i / 8, b = i % 8;
      if (i % 8 == 2) {
        asm volatile("s_add_u32 m0, %3, %4\n\t"
                     "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                     "buffer_load_dwordx4 %5, %6, %7 offen lds"
                     : "+a"(acc[a][b])
                     : "v"(fw[H][b]), "v"(fr[H][a]), "s"(dst), "n"(i / 8 * 4096),
                       "v"(off[i / 8]), "s"(rs), "s"(k0)
                     : "m0", "scc", "memory");
      } else {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[a][b]) : "v"(fw[H][b]), "v"(fr[H][a]));
      }
      if (i < 32 && i % 2 == 1) {
        const int j = i / 2;
        __builtin_amdgcn_sched_barrier(0);
        if (j < 8)
          fw[H ^ 1][j] = *reinterpret_cast<const u32x4*>(wnx + j * 16 * WT_K);
        else
          fr[H ^ 1][j - 8] =
              *reinterpret_cast<const u32x4*>(rn + (j - 8) * 16 * WT_K);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
      for (int b = 0; b < 8; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_nop 7" ::: "memory");
    const Place p = place(round);
#pragma unroll 1
    for (int s = 0; s < p.n; ++s) {
      const int next = bw == 2 ? 0 : bw + 1, over = bw == 0 ? 2 : bw - 1;
      half(wt_int<0>{}, rl + bx * WT_BUF + at1, wl + bw * WT_BUF + at1, rw,
           to + (2 + over) * WT_BYTES, ow);
      // the next step is there: behind its loads only the weights of the one after
      // were asked for, and at the start of a tile the stores of the one before
      if (s == 0 && round > 0)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 + STORES) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      half(wt_int<1>{}, rl + (bx ^ 1) * WT_BUF + at0, wl + next * WT_BUF + at0, rx,
           to + bx * WT_BYTES, ox);
      advance();
      bx ^= 1;
      bw = next;
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

    // acc[a][b][j]: column 4 lg + j of tile b, row lc of tile a
    constexpr unsigned SIZE = OUT == PARTS ? 4 : 2;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (char*)out_ + (((long)p.part * M + p.m0) * N + p.n0) * SIZE, 0,
        ((unsigned)min(WT_ROWS, M - p.m0) - 1) * (unsigned)N * SIZE +
            (unsigned)min(COLS, N - p.n0) * SIZE,
        0x00020000);
    unsigned row = (unsigned)(wm * 128 + lc) * (unsigned)N * SIZE;
    asm volatile("" : "+v"(row));           // not a register for every row
#pragma unroll
    for (int a = 0; a < 8; ++a) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < HC / 16; b += 2) {
        // columns and rows beyond the result are not stored
        const int col = wn * HC + b * 16 + lg * 8;
        const unsigned off = p.n0 + col < N ? row + (unsigned)a * 16u * SIZE * (unsigned)N +
                                                  col * SIZE
                                            : 0xffffff00u;
        if constexpr (OUT == PARTS) {
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              o[j] = __builtin_bit_cast(unsigned, wt_sum(acc[a][b + i][j]));
            __builtin_amdgcn_raw_buffer_store_b128(
                o, ro, p.n0 + col < N ? off + i * 16 : 0xffffff00u, 0, 0);
          }
        } else {
          u32x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int e = j % 2 * 2;
            const f32x4 g = acc[a][b + j / 2];
            const f32x4 u = acc[a][b + 4 + j / 2];
            o[j] = wt_pack(wt_silu(wt_sum(g[e]), wt_sum(u[e])),
                           wt_silu(wt_sum(g[e + 1]), wt_sum(u[e + 1])));
          }
          __builtin_amdgcn_raw_buffer_store_b128(o, ro, off, 0, 0);
        }
      }
    }
  }
  // no load is left that would write to the LDS of a later workgroup
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace

// x [M, K] of row stride xs; offsets inside a tile's operands are 32 bits of bytes.
// splits 0: the activation of the product (w [2 N, K]), else the product in fp32 parts,
// each of two steps of k or more.
void wide_launch(void* out, const void* x, const void* w, int M, int N, int K, long xs,
                 int splits, int* err_unsupported, hipStream_t s) {
  const long far = 1l << 32, wn = splits == 0 ? 2l * N : N;
  *err_unsupported = K % WT_K != 0 || K < 2 * WT_K || N % 8 != 0 ||
                     (wn + WT_ROWS) * K * 2 >= far || (xs + K) * WT_ROWS * 2 >= far ||
                     4l * N * (WT_ROWS + 1) >= far - 256 || splits < 0 ||
                     (splits > 0 && K / WT_K / splits < 2);
  if (*err_unsupported || M == 0 || N == 0) return;
#define WIDE(OUT)                                                               \
  hipLaunchKernelGGL(wide_kernel<OUT>, dim3(WT_CUS), dim3(256), 0, s, out,      \
                     (const unsigned short*)x, (const unsigned short*)w, M, N, K, xs, \
                     splits)
  if (splits == 0) WIDE(SILU);
  else WIDE(PARTS);
#undef WIDE
}
