// Products of many rows for MI355X (gfx950) in tiles of up to 256 rows and 256 weight
// rows: x W^T, silu(x Wg^T) * (x Wu^T) in one launch, or x W^T cut over k.
//
// One workgroup a CU walks its tiles; four waves of up to 128 x 128 on
// mfma_f32_16x16x32_bf16 (of random numbers 2.1 PFLOP/s before the card's power
// limits it, 32x32x16 1.85), fp32 sums in the accumulation registers. Larger waves
// read less: 64 x 64 ask the LDS for 128 bytes a cycle at the full matrix rate, which
// is all that it has, 128 x 128 for 64, and the L1 for 32 where tiles of 128 x 128 ask
// it for the 64 that it has.
// But 256 workgroups work in rounds of tiles, and where a round of 256 x 256 stays half
// empty a smaller tile costs less than it fills: the caller chooses. In rounds that are
// full, tiles of 256 x 256 reach 1.00, x 224 .98, x 192 .97, x 160 .93, x 128 .88, 192 x
// 256 .97, x 192 .92, 128 x 192 .78, x 128 .68, x 64 .50 of the rate, from 1024 to 14336
// k, weights out of HBM.
// A step is 64 k: rows of 128 bytes, 16-byte chunk c of row r at c ^ (r / 2 % 8), which
// 16 rows of one chunk read without conflict. (Rows of 32 k, five steps deep: 1530 us
// where these take 1390, 8192 rows of 28672 x 4096; the L1 serves half lines.) Two to
// five buffers of rows and one more of weights fill the LDS; buffers of a step are asked
// for as many steps ahead, through the end of a tile into the next one, whose first steps
// come while the results of this one are stored.
// With one wave a SIMD the matrix unit idles whenever the wave issues more than two or
// three other instructions between two products: operands are read half a step ahead,
// and each gap between products holds one LDS read or one load, no branch (8 loads
// behind every eighth product 1390 us, one in every eighth gap 1310).
// The products are inline asm that adds in place: left to itself the compiler writes
// them to other registers and copies, all 256 being taken. It does not see the products
// in the asm, so the waits before their results are read stand here (s_nop), and a loop
// of one body keeps it from copying them in between.
// With the activation, 28672 x 4096: 8192 rows 1278 us (1505 TFLOP/s), 2039 rows 341 in
// tiles of 256 x 224 (256 x 256, whose last round is half empty, 354), 512 rows out of
// HBM 91 (94); the library's product and the activation behind it 1290 + 127, 353 + 31,
// 97 + 11. Without: 2039 rows of 6144 x 4096 in tiles of 256 x 192 75 (library 84), of
// 4096 x 4096 in 256 x 128 56 (62); 4188 of 2048 x 4096 in 192 x 192 58 (65). Where
// whole tiles of 256 x 256 fill the rounds it is the library's own tile, .91 to 1.1 of
// its time.
// Products whose consumer adds fp32 parts up fill the workgroups cut over k: with an RMS
// norm behind, 4096 x 14336 at 512 rows 66 us (before 73), 640 84 (143), 1024 107 (159),
// 2039 197 (217); 512 rows of 6144 x 4096 42 (49), of 4096 x 4096 33 (38).
#include "wide_tiles.h"

namespace {

typedef __attribute__((ext_vector_type(2))) unsigned u32x2;

constexpr int WT_K = 64;
constexpr int WT_CUS = 256;                 // workgroups of a launch

// SILU: out [M, N] = silu(x Wg^T) * (x Wu^T), w [2 N, K] = Wg, then Wu. ROWS: out
// [M, N] = x W^T, w [N, K]. PARTS: out [splits, M, N] of it in fp32, each of its own
// steps of k.
enum WideOut { SILU, ROWS, PARTS };

// A wave has RF x CF tiles of 16 rows and 16 weight rows, the workgroup 2 x 2 waves.
template <int OUT, int RF, int CF>
__global__ __launch_bounds__(256, 1) void wide_kernel(
    void* __restrict__ out_, const unsigned short* __restrict__ x,
    const unsigned short* __restrict__ w, int M, int N, int K, long xs, int splits) {
  constexpr int MT = 32 * RF, WT = 32 * CF; // rows and weight rows of a tile
  constexpr int COLS = OUT == SILU ? WT / 2 : WT;            // columns of a tile
  constexpr int HC = COLS / 2;              // of a wave
  // buffers of the rows; of the weights there is one more
  constexpr int NR = 5 * RF + 6 * CF <= 40 ? 5 : 4 * RF + 5 * CF <= 40 ? 4
                   : 3 * RF + 4 * CF <= 40 ? 3 : 2;
  constexpr int NW = NR + 1;
  // loads behind the last one of the next step, halfway through a step
  constexpr int BEHIND = CF * (NR - 1) + RF * (NR - 2);
  // tiles side by side of which a lane's columns are neighbours: 16 bytes of the result
  constexpr int GROUP = OUT == SILU ? 4 : 2, EACH = OUT == SILU ? 2 : 4;
  constexpr int WHOLE = CF / GROUP, REST = CF % GROUP;
  // stores of a wave at the end of a tile, as far as a wait can count them
  constexpr int ALL = RF * (OUT == PARTS ? CF : WHOLE + (REST != 0));
  constexpr int STORES = ALL < 63 - BEHIND ? ALL : 63 - BEHIND;
  constexpr int XB = MT * WT_K, WB = WT * WT_K;              // elements of a buffer
  __shared__ __attribute__((aligned(16))) unsigned short lds[NR * XB + NW * WB];
  const int tid = threadIdx.x, lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave >> 1, wn = wave & 1;
  const int lc = lane & 15, lg = lane >> 4;
  const int steps = K / WT_K;
  const int WN = OUT == SILU ? 2 * N : N;   // weight rows
  const int mt = (M + MT - 1) / MT, nt = (N + COLS - 1) / COLS;

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
    p.m0 = one((g * 8 + in % high) * MT);
    p.n0 = one(in / high * COLS);
    return p;
  };

  // A wave's load i brings rows (i * 4 + wave) * 8 .. of 128 bytes to the LDS. Rows
  // 4 g .. of a group of tiles are neighbouring columns, those of the lanes of g. Of
  // SILU two tiles are the gate's, two the up product's; where no four are left, rows 0
  // and 1 of each four the gate's.
  unsigned ox[RF], ow[CF];
#pragma unroll
  for (int i = 0; i < RF || i < CF; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    const int at = ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    if (i < RF) ox[i] = ((unsigned)row * (unsigned)xs + at) * 2;
    if (i < CF) {
      const int b = (row >> 4) % CF, g = (row >> 2) & 3, j = row & 3;
      int col = row / (CF * 16) * HC + b / GROUP * 32;
      if (b >= WHOLE * GROUP)               // REST of them
        col += OUT == SILU ? g * REST * 2 + b % GROUP * 2 + (j & 1) + (j & 2 ? N : 0)
                           : g * REST * 4 + b % GROUP * 4 + j;
      else
        col += g * 8 + (b & 1) * 4 + j + (OUT == SILU && b & 2 ? N : 0);
      ow[i] = ((unsigned)col * (unsigned)K + at) * 2;
    }
  }
  const int at0 = lc * WT_K + (lg ^ ((lc >> 1) & 7)) * 8, at1 = at0 ^ 32;
  const unsigned short* rl = lds + wm * (XB / 2);
  const unsigned short* wl = lds + NR * XB + wn * (WB / 2);
  const unsigned to = lds_address(lds) + wave * 8 * WT_K * 2;

  // The step that is loaded next: of the tile of round `lr`, with `left` steps to come;
  // k0: its bytes from the start of a row. Weight rows lie a power of two apart, and
  // workgroups at one place of theirs meet on a few memory channels: each eighth of the
  // columns, about an XCD's, begins an eighth of the row further on (512 rows of 28672 x
  // 4096 out of HBM 97 -> 91 us; each column tile at a place of its own 96, and 1327 for
  // 1250 at 8192 rows, whose rows then miss the L2). A column's rows all begin at one
  // place: equal ones get equal sums. Of no use in more rows, which compute longer than
  // they load (7122 x 8192 x 2048 330 -> 331), and parts begin elsewhere anyway.
  auto turn = [&](const Place& p) {
    return OUT != PARTS && M <= 2048 ? one(p.n0 / COLS * 8 / nt * steps / 8) : p.from;
  };
  int lr = 0, left = 0;
  unsigned k0 = 0;
  i32x4 rx{}, rw{};
  auto point = [&]() {
    if (lr < rounds) {
      const Place p = place(lr);
      left = p.n;
      k0 = (unsigned)turn(p) * (WT_K * 2);
      rx = wt_rsrc(x + p.m0 * xs, ((unsigned)min(MT, M - p.m0) - 1) *
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
    if (OUT != PARTS && k0 == (unsigned)K * 2) k0 = 0;
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
  for (int s = 0; s < NR; ++s) {
#pragma unroll
    for (int i = 0; i < CF; ++i) load(to + (NR * XB + s * WB) * 2 + i * 4096, ow[i], rw);
#pragma unroll
    for (int i = 0; i < RF; ++i) load(to + s * XB * 2 + i * 4096, ox[i], rx);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NR - 1) * (RF + CF)) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int bx = 0, bw = 0;                       // buffers of the step at hand

  u32x4 fr[2][RF], fw[2][CF];
#pragma unroll
  for (int i = 0; i < CF; ++i)
    fw[0][i] = *reinterpret_cast<const u32x4*>(wl + at0 + i * 16 * WT_K);
#pragma unroll
  for (int i = 0; i < RF; ++i)
    fr[0][i] = *reinterpret_cast<const u32x4*>(rl + at0 + i * 16 * WT_K);
  f32x4 acc[RF][CF];

  // The products of half `h` of a step; into the gaps between them go the operands of
  // the next half, from rn and wnx, and the loads to `dst`: of weights, then of rows.
  auto half = [&](auto h, const unsigned short* rn, const unsigned short* wnx,
                  const i32x4& rs, unsigned dst, const unsigned* off) {
    constexpr int H = decltype(h)::value;
    constexpr int P = RF * CF, LOADS = H == 0 ? CF : RF, READS = RF + CF;
    constexpr int EVERY = P / LOADS, FIRST = EVERY > 2 ? 2 : 1;
    constexpr int GAP = 2 * READS + 8 <= P ? 2 : 1;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int a = i / CF, b = i % CF, at = (i - FIRST) / EVERY;
      if (i >= FIRST && (i - FIRST) % EVERY == 0 && at < LOADS) {
        asm volatile("s_add_u32 m0, %3, %4\n\t"
                     "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                     "buffer_load_dwordx4 %5, %6, %7 offen lds"
                     : "+a"(acc[a][b])
                     : "v"(fw[H][b]), "v"(fr[H][a]), "s"(dst), "n"(at * 4096),
                       "v"(off[at]), "s"(rs), "s"(k0)
                     : "m0", "scc", "memory");
      } else {
        asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                     : "+a"(acc[a][b]) : "v"(fw[H][b]), "v"(fr[H][a]));
      }
      if (i % GAP == GAP - 1 && i / GAP < READS) {
        const int j = i / GAP;
        __builtin_amdgcn_sched_barrier(0);
        if (j < CF)
          fw[H ^ 1][j] = *reinterpret_cast<const u32x4*>(wnx + j * 16 * WT_K);
        else
          fr[H ^ 1][j - CF] =
              *reinterpret_cast<const u32x4*>(rn + (j - CF) * 16 * WT_K);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
#pragma unroll
    for (int a = 0; a < RF; ++a)
#pragma unroll
      for (int b = 0; b < CF; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_nop 7" ::: "memory");
    const Place p = place(round);
#pragma unroll 1
    for (int s = 0; s < p.n; ++s) {
      const int nx = bx == NR - 1 ? 0 : bx + 1;
      const int nw = bw == NW - 1 ? 0 : bw + 1, over = bw == 0 ? NW - 1 : bw - 1;
      half(wt_int<0>{}, rl + bx * XB + at1, wl + bw * WB + at1, rw,
           to + (NR * XB + over * WB) * 2, ow);
      // the next step is there: BEHIND loads came after its own, and where those were
      // asked for in the tile before, its stores
      if (s < NR - 1 && round > 0)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND + STORES) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      half(wt_int<1>{}, rl + nx * XB + at0, wl + nw * WB + at0, rx, to + bx * XB * 2, ox);
      advance();
      bx = nx;
      bw = nw;
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

    // acc[a][b][j]: row 4 lg + j of weight tile b, row lc of tile a
    constexpr unsigned SIZE = OUT == PARTS ? 4 : 2;
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        (char*)out_ + (((long)p.part * M + p.m0) * N + p.n0) * SIZE, 0,
        ((unsigned)min(MT, M - p.m0) - 1) * (unsigned)N * SIZE +
            (unsigned)min(COLS, N - p.n0) * SIZE,
        0x00020000);
    unsigned row = (unsigned)(wm * (MT / 2) + lc) * (unsigned)N * SIZE;
    asm volatile("" : "+v"(row));           // not a register for every row
#pragma unroll
    for (int a = 0; a < RF; ++a) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int b = 0; b < CF; b += GROUP) {
        const int side = CF - b < GROUP ? REST : GROUP;
        // columns and rows beyond the result are not stored; N is a multiple of 8
        const int col = wn * HC + b / GROUP * 32 + lg * side * EACH;
        const unsigned off = row + (unsigned)a * 16u * SIZE * (unsigned)N + col * SIZE;
        if constexpr (OUT == PARTS) {
#pragma unroll
          for (int i = 0; i < side; ++i) {
            u32x4 o;
#pragma unroll
            for (int j = 0; j < 4; ++j)
              o[j] = __builtin_bit_cast(unsigned, wt_sum(acc[a][b + i][j]));
            __builtin_amdgcn_raw_buffer_store_b128(
                o, ro, p.n0 + col + i * 4 < N ? off + i * 16 : 0xffffff00u, 0, 0);
          }
        } else {
          u32x4 o{};                        // two columns each
#pragma unroll
          for (int j = 0; j < side * EACH / 2; ++j) {
            if constexpr (OUT == SILU) {
              const bool all = side == GROUP;
              const f32x4 g = acc[a][all ? b + j / 2 : b + j];
              const f32x4 u = acc[a][all ? b + 2 + j / 2 : b + j];
              const int at = all ? j % 2 * 2 : 0, up = all ? at : 2;
              o[j] = wt_pack(wt_silu(wt_sum(g[at]), wt_sum(u[up])),
                             wt_silu(wt_sum(g[at + 1]), wt_sum(u[up + 1])));
            } else {
              const f32x4 v = acc[a][b + j / 2];
              o[j] = wt_pack(wt_sum(v[j % 2 * 2]), wt_sum(v[j % 2 * 2 + 1]));
            }
          }
          const int words = side * EACH / 2, end = N - p.n0 - col;
          if (words == 4)
            __builtin_amdgcn_raw_buffer_store_b128(o, ro, end > 0 ? off : 0xffffff00u, 0, 0);
          else if (words == 2)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{o[0], o[1]}, ro,
                                                  end > 0 ? off : 0xffffff00u, 0, 0);
          else                              // of SILU; N may end within it
#pragma unroll
            for (int j = 0; j < words; ++j)
              __builtin_amdgcn_raw_buffer_store_b32(
                  o[j], ro, end > 2 * j ? off + j * 4 : 0xffffff00u, 0, 0);
        }
      }
    }
  }
  // no load is left that would write to the LDS of a later workgroup
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace

// kind 0: silu(gate) * up, w [2 N, K]; 1: the product; 2: in fp32 parts, each of two
// steps of k or more. rf, cf: a quarter of the tile in 16 rows and weight rows. x [M, K]
// of row stride xs; offsets inside a tile's operands are 32 bits of bytes.
void wide_launch(int kind, void* out, const void* x, const void* w, int M, int N, int K,
                 long xs, int splits, int rf, int cf, int* err_unsupported,
                 hipStream_t s) {
  constexpr int MOST = 256;
  const long far = 1l << 32, wn = kind == 0 ? 2l * N : N;
  *err_unsupported = K % WT_K != 0 || K < 2 * WT_K || N % 8 != 0 ||
                     (wn + MOST) * K * 2 >= far || (xs + K) * MOST * 2 >= far ||
                     4l * N * (MOST + 1) >= far - 256 || splits < 1 ||
                     K / WT_K / splits < 2 || kind < 0 || kind > 2 || rf < 0 || rf > 9 ||
                     cf < 0 || cf > 9;
  if (*err_unsupported || M == 0 || N == 0) return;
  switch (kind * 100 + rf * 10 + cf) {
#define WIDE(OUT, RF, CF)                                                              \
    case OUT * 100 + RF * 10 + CF:                                                     \
      hipLaunchKernelGGL((wide_kernel<OUT, RF, CF>), dim3(WT_CUS), dim3(256), 0, s,    \
                         out, (const unsigned short*)x, (const unsigned short*)w, M, N, \
                         K, xs, splits);                                               \
      break
    WIDE(SILU, 8, 8); WIDE(SILU, 8, 7); WIDE(SILU, 8, 6); WIDE(SILU, 8, 5);
    WIDE(SILU, 8, 4); WIDE(SILU, 6, 8);
    WIDE(ROWS, 8, 7); WIDE(ROWS, 8, 6); WIDE(ROWS, 8, 4); WIDE(ROWS, 6, 8);
    WIDE(ROWS, 6, 6); WIDE(ROWS, 4, 6); WIDE(ROWS, 4, 4); WIDE(ROWS, 4, 2);
    WIDE(PARTS, 8, 8); WIDE(PARTS, 8, 6); WIDE(PARTS, 8, 4); WIDE(PARTS, 6, 8);
    WIDE(PARTS, 6, 6); WIDE(PARTS, 4, 6); WIDE(PARTS, 4, 4);
#undef WIDE
    default: *err_unsupported = 1;
  }
}
