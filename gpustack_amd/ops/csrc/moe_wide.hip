// Expert products of many rows for MI355X (gfx950): the two products of moe_gemm.hip
// in tiles of up to 320 rows of an expert and 192 weight rows.
//
// The loop is that of wide_tiles.hip: one workgroup a CU walks its tiles, four waves,
// one a SIMD, operands half a step ahead, loads two steps ahead and on into the next
// tile, products that add in place in inline asm, one other instruction to a gap.
// Experts' weights come out of memory once; at 250 rows an expert that stream takes
// about as long as the products. So a tile has to hold all rows of an expert, or its
// weights are read and waited for twice; 320 rows of 192 weight rows are what the 256
// accumulation registers of a lane hold (240), two buffers of rows and three of weights
// what the LDS does (152 KB). More rows are parts of one size. A wave has half of the
// rows and half of the weights; a tile of fewer rows runs a loop of as many products as
// its 64 rows ask for.
// Of gate and up a wave has 48 rows each, of the same columns; of down 96, row 4 g + j
// of tiles 2 p and 2 p + 1 is column 32 p + 8 g + j and + 4, so that a lane stores 16
// bytes and four lanes 64.
// An XCD's tiles follow each other by expert, columns, parts: its L2 reads an expert's
// rows once for all of them.
// Bound by the weight stream, the products and the end of a tile (4 to 6 us, in which
// no load leaves) one behind the other: a wave waits for its loads in their order, so
// two steps ahead of the rows is as far as the weights get. 128 experts of 1536 +
// 2048 x 2048 + 768 at 254 rows each: 202 + 153 us, 141 + 100 without the memory, 165
// + 111 without the loads (tiles of 128: 283 + 180); 188 rows 187 + 133 (232 + 149); 8
// of 4096 x 14336 at 1024 rows 1630 + 830 (2160 + 1200), 1170 TFLOP/s.
// Tried: the loads of a step in one half, weights a step further ahead 1600 -> 1680;
// tiles of every 32 rows no faster; whole parts of 320 and a rest, large ones dealt
// first: even at 254 rows, 250 -> 266 at 500.
#include "wide_tiles.h"

namespace {

constexpr int MW_ROWS = 320, MW_W = 192, MW_K = 64;
constexpr int MW_XBUF = MW_ROWS * MW_K, MW_WBUF = MW_W * MW_K;   // elements
constexpr int MW_XL = MW_ROWS / 32, MW_WL = MW_W / 32;           // loads of a wave
constexpr int MW_TILES = MW_W / 32;        // weight tiles of a wave
constexpr int MW_CUS = 256;
constexpr int MW_EXPERTS = 256;            // a lane keeps four of them
constexpr unsigned MW_NOWHERE = 0xffffff00u;

template <bool DOWN>
__global__ __launch_bounds__(256, 1) void moe_wide_kernel(
    unsigned short* __restrict__ out,        // act [TK, I] | contrib [TK, H]
    const unsigned short* __restrict__ src,  // x [T, H] | act [TK, I]
    const unsigned short* __restrict__ w,    // [E, 2I, H] | [E, H, I]
    const int* __restrict__ rows,            // s_tok | order, [TK]
    const float* __restrict__ s_w,           // DOWN: routing weights, sorted
    const int* __restrict__ offs, const int* __restrict__ counts, int E, int N,
    int K, unsigned src_bytes, unsigned out_bytes) {
  constexpr int OW = DOWN ? MW_W : MW_W / 2;  // columns of a tile
  constexpr int HW = OW / 2;                  // of a wave
  __shared__ __attribute__((aligned(16))) unsigned short
      lds[2 * MW_XBUF + 3 * MW_WBUF];
  const int tid = threadIdx.x, lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave >> 1, wn = wave & 1;
  const int lc = lane & 15, lg = lane >> 4;
  const int n = K / MW_K, nnt = (N + OW - 1) / OW;

  // lane l keeps experts l, l + 64 ..: rows, first row, parts up to and with it
  int cnt[4], first_of[4], upto[4], total = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int e = j * 64 + lane;
    cnt[j] = e < E ? counts[e] : 0;
    first_of[j] = e < E ? offs[e] : 0;
    int p = (cnt[j] + MW_ROWS - 1) / MW_ROWS;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
      const int before = __shfl_up(p, m, 64);
      if (lane >= m) p += before;
    }
    upto[j] = total + p;
    total += __builtin_amdgcn_readlane(p, 63);
  }
  const int items = total * nnt;
  const int xcd = blockIdx.x & 7, per = MW_CUS / 8, slot = blockIdx.x >> 3;
  const int q = items / 8, r = items % 8;
  const int count = xcd < r ? q + 1 : q;     // tiles of this XCD
  const int start = xcd * q + min(xcd, r);
  if (slot >= count) return;
  const int rounds = (count - slot + per - 1) / per;

  struct Place { int n0, first, rows, e, turn; };
  auto place = [&](int round) {              // divisions: once a tile
    const int item = start + round * per + slot, part_at = item / nnt;
    int e = 0, c = 0, f = 0, u = 0;
    bool found = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const unsigned long more = __ballot(upto[j] > part_at);
      if (!found && more != 0) {
        const int l = __builtin_ctzl(more);
        found = true;
        e = j * 64 + l;
        c = __builtin_amdgcn_readlane(cnt[j], l);
        f = __builtin_amdgcn_readlane(first_of[j], l);
        u = __builtin_amdgcn_readlane(upto[j], l);
      }
    }
    auto one = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int parts = (c + MW_ROWS - 1) / MW_ROWS;
    const int local = item - (u - parts) * nnt;
    const int high = (c + parts - 1) / parts, from = local % parts * high;
    // Weight rows lie a power of two apart: workgroups that all read the same k of
    // theirs meet on a few memory channels, so each expert begins elsewhere, its
    // workgroups in one place (188 rows of each of 128 187 us -> 182, 64 157 -> 148).
    // The second product's rows are short, and it gains nothing.
    return Place{one(local / parts * OW), one(f + from), one(min(high, c - from)),
                 one(e), DOWN ? 0 : one((e * 7 + e / 16) % n)};
  };

  // A wave's load i brings rows (i * 4 + wave) * 8 .. of 128 bytes, 16-byte chunk c of
  // row r to c ^ (r / 2 % 8).
  const int at_k = ((lane & 7) ^ ((lane >> 4) & 3) ^ ((wave & 1) << 2)) * 8;
  unsigned ox[MW_XL], ow[MW_WL];
  int nx[MW_XL];                             // rows of x of the tile after the loaded
#pragma unroll
  for (int i = 0; i < MW_WL; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    const int in = row % 96, b = in / 16, g = in >> 2 & 3, j = in & 3;
    const int col = row / 96 * HW +
                    (DOWN ? b / 2 * 32 + g * 8 + b % 2 * 4 + j
                          : b % 3 * 16 + in % 16 + (b >= 3 ? N : 0));
    ow[i] = ((unsigned)col * (unsigned)K + at_k) * 2;
  }
  auto x_row = [&](int i) { return (i * 4 + wave) * 8 + lane / 8; };
  auto gather = [&](const Place& p) {        // tokens of a tile's rows
#pragma unroll
    for (int i = 0; i < MW_XL; ++i) {
      const int at = x_row(i);
      nx[i] = rows[p.first + min(at, p.rows - 1)];
    }
  };
  auto arrived = [&]() {                     // here, not where they are used
#pragma unroll
    for (int i = 0; i < MW_XL; ++i) asm volatile("" : "+v"(nx[i]));
  };

  // The step that is loaded next: lk of the tile of round `lr`, which is the one at
  // hand or the next.
  int lr = 0, lk = 0;
  unsigned k0 = 0;                           // its bytes from the start of a row
  i32x4 rx{}, rw{};
  Place cur = place(0), nxt = rounds > 1 ? place(1) : cur;
  auto point = [&](const Place& p) {
    k0 = (unsigned)p.turn * (MW_K * 2);
    if (lr < rounds) {
      rw = wt_rsrc(w + ((long)p.e * (DOWN ? N : 2 * N) + p.n0) * K,
                   (unsigned)((DOWN ? N : 2 * N) - p.n0) * (unsigned)K * 2);
      if constexpr (DOWN) {
        rx = wt_rsrc(src + (long)p.first * K, (unsigned)p.rows * (unsigned)K * 2);
      } else {
#pragma unroll
        for (int i = 0; i < MW_XL; ++i)
          ox[i] = x_row(i) < p.rows ? ((unsigned)nx[i] * (unsigned)K + at_k) * 2
                                    : MW_NOWHERE;
      }
    } else {
      rx[2] = rw[2] = 0;
    }
  };
  auto advance = [&]() {
    if (++lk == n) {
      lk = 0;
      ++lr;
      point(nxt);
    } else {
      k0 += MW_K * 2;
      if (k0 == (unsigned)K * 2) k0 = 0;
    }
  };
  const unsigned to = lds_address(lds) + wave * 8 * MW_K * 2;
  auto load = [&](unsigned at, unsigned off, const i32x4& rs) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                 "buffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(at), "v"(off), "s"(rs), "s"(k0)
                 : "m0", "memory");
  };
  // DOWN: result row and weight of this lane's row of each tile of a wave's rows
  int orow[MW_XL], next_row[MW_XL];
  float rwt[MW_XL], next_w[MW_XL];
  auto height = [&](const Place& p) { return (p.rows + 63) / 64 * 2; };
  auto results = [&](const Place& p) {
    const int nb = height(p);
#pragma unroll
    for (int a = 0; a < MW_XL; ++a) {
      const int at = p.first + min((wm * nb + a) * 16 + lc, p.rows - 1);
      next_row[a] = rows[at];
      next_w[a] = s_w[at];
    }
  };
  auto results_arrived = [&]() {
#pragma unroll
    for (int a = 0; a < MW_XL; ++a) {
      asm volatile("" : "+v"(next_row[a]), "+v"(next_w[a]));
      orow[a] = next_row[a];
      rwt[a] = next_w[a];
    }
  };

  if constexpr (DOWN) {
#pragma unroll
    for (int i = 0; i < MW_XL; ++i)
      ox[i] = ((unsigned)x_row(i) * (unsigned)K + at_k) * 2;
    results(cur);
    results_arrived();
    point(cur);
  } else {
    rx = wt_rsrc(src, src_bytes);
    gather(cur);
    arrived();
    point(cur);
    gather(nxt);
    arrived();
  }
  constexpr unsigned XB = MW_XBUF * 2, WB = MW_WBUF * 2, W0 = 2 * XB;   // bytes
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < MW_WL; ++i) load(to + W0 + s * WB + i * 4096, ow[i], rw);
#pragma unroll
    for (int i = 0; i < MW_XL; ++i) load(to + s * XB + i * 4096, ox[i], rx);
    advance();
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MW_XL + MW_WL) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  const int at0 = lc * MW_K + (lg ^ ((lc >> 1) & 7)) * 8, at1 = at0 ^ 32;
  const unsigned short* wl = lds + 2 * MW_XBUF + wn * (MW_W / 2) * MW_K;
  int bx = 0, bw = 0;                        // buffers of the step at hand
  int stores = 0;                            // of the tile before, at least

  // A tile whose waves have NB * 16 rows each.
  auto tile = [&](auto nb, int round) {
    constexpr int NB = decltype(nb)::value, NW = MW_TILES;
    constexpr int GAPS = NB * NW, READS = NB + NW;
    constexpr int SPAN = READS > GAPS / 2 ? READS : GAPS / 2;  // gaps with reads
    const unsigned short* rl = lds + wm * NB * 16 * MW_K;
    f32x4 acc[NB][NW];
    u32x4 fr[2][NB], fw[2][NW];
#pragma unroll
    for (int i = 0; i < NW; ++i)
      fw[0][i] =
          *reinterpret_cast<const u32x4*>(wl + bw * MW_WBUF + at0 + i * 16 * MW_K);
#pragma unroll
    for (int i = 0; i < NB; ++i)
      fr[0][i] =
          *reinterpret_cast<const u32x4*>(rl + bx * MW_XBUF + at0 + i * 16 * MW_K);
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int b = 0; b < NW; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_nop 7" ::: "memory");

    // The products of half `h` of a step; into the gaps between them go the operands
    // of the next half, from rn and wnx, and `loads` loads to `dst`.
    auto half = [&](auto h, auto loads, const unsigned short* rn,
                    const unsigned short* wnx, const i32x4& rs, unsigned dst,
                    const unsigned* off) {
      constexpr int H = decltype(h)::value, L = decltype(loads)::value;
      int read = 0, ld = 0;
#pragma unroll
      for (int i = 0; i < GAPS; ++i) {
        const int a = i / NW, b = i % NW;
        if (ld < L && i == (2 * ld + 1) * GAPS / (2 * L)) {
          asm volatile("s_add_u32 m0, %3, %4\n\t"
                       "v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                       "buffer_load_dwordx4 %5, %6, %7 offen lds"
                       : "+a"(acc[a][b])
                       : "v"(fw[H][b]), "v"(fr[H][a]), "s"(dst), "n"(ld * 4096),
                         "v"(off[ld]), "s"(rs), "s"(k0)
                       : "m0", "scc", "memory");
          ++ld;
        } else {
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0"
                       : "+a"(acc[a][b]) : "v"(fw[H][b]), "v"(fr[H][a]));
        }
        if (read < READS && i == read * SPAN / READS) {
          __builtin_amdgcn_sched_barrier(0);
          if (read < NW)
            fw[H ^ 1][read] =
                *reinterpret_cast<const u32x4*>(wnx + read * 16 * MW_K);
          else
            fr[H ^ 1][read - NW] =
                *reinterpret_cast<const u32x4*>(rn + (read - NW) * 16 * MW_K);
          __builtin_amdgcn_sched_barrier(0);
          ++read;
        }
      }
    };
#pragma unroll 1
    for (int s = 0; s < n; ++s) {
      const int next = bw == 2 ? 0 : bw + 1, last = bw == 0 ? 2 : bw - 1;
      half(wt_int<0>{}, wt_int<MW_WL>{}, rl + bx * MW_XBUF + at1,
           wl + bw * MW_WBUF + at1, rw, to + W0 + last * WB, ow);
      // the next step is there: behind its loads only the weights of the one after
      // were asked for, and at the start of a tile the stores of the one before
      if (s == 0 && stores >= 24)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(MW_WL + 24) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(MW_WL) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      half(wt_int<1>{}, wt_int<MW_XL>{}, rl + (bx ^ 1) * MW_XBUF + at0,
           wl + next * MW_WBUF + at0, rx, to + bx * XB, ox);
      advance();
      bx ^= 1;
      bw = next;
    }
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");

    // what the tiles ahead need of the routing comes while this one is stored
    const Place far = round + 2 < rounds ? place(round + 2) : nxt;
    if constexpr (DOWN) results(nxt);
    else gather(far);
    // acc[a][b][j]: row lc of tile a, weight row 4 lg + j of tile b
    const Place p = cur;
    const int col0 = p.n0 + wn * HW + lg * (DOWN ? 8 : 4);
    const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
        DOWN ? out : out + (long)p.first * N, 0,
        DOWN ? out_bytes : (unsigned)p.rows * (unsigned)N * 2, 0x00020000);
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      __builtin_amdgcn_sched_barrier(0);
      const int row = (wm * NB + a) * 16 + lc;
      const unsigned at =
          ((unsigned)(DOWN ? orow[a] : row) * (unsigned)N + (unsigned)col0) * 2;
      const bool in = row < p.rows;
      if constexpr (DOWN) {
#pragma unroll
        for (int b = 0; b < NW; b += 2) {
          u32x4 o;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const f32x4 v = acc[a][b + j / 2];
            const int e = j % 2 * 2;
            o[j] = wt_pack(wt_sum(v[e]) * rwt[a], wt_sum(v[e + 1]) * rwt[a]);
          }
          __builtin_amdgcn_raw_buffer_store_b128(
              o, ro, in && col0 + b * 16 < N ? at + b * 32 : MW_NOWHERE, 0, 0);
        }
      } else {
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const f32x4 g = acc[a][b], u = acc[a][b + 3];
          __attribute__((ext_vector_type(2))) unsigned o;
#pragma unroll
          for (int j = 0; j < 2; ++j)
            o[j] = wt_pack(wt_silu(wt_sum(g[2 * j]), wt_sum(u[2 * j])),
                           wt_silu(wt_sum(g[2 * j + 1]), wt_sum(u[2 * j + 1])));
          __builtin_amdgcn_raw_buffer_store_b64(
              o, ro, in && col0 + b * 16 < N ? at + b * 32 : MW_NOWHERE, 0, 0);
        }
      }
    }
    stores = NB * 3;
    cur = nxt;
    nxt = far;
    if constexpr (DOWN) results_arrived();
    else arrived();
  };
#pragma unroll 1
  for (int round = 0; round < rounds; ++round) {
    switch (height(cur)) {
      case 2: tile(wt_int<2>{}, round); break;
      case 4: tile(wt_int<4>{}, round); break;
      case 6: tile(wt_int<6>{}, round); break;
      case 8: tile(wt_int<8>{}, round); break;
      default: tile(wt_int<10>{}, round); break;
    }
  }
  // no load is left that would write to the LDS of a later workgroup
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace

// Offsets inside an operand of a tile are 32 bits of bytes; of x, of an expert's weights
// and of contrib it is all of it.
bool moe_wide_takes(int down, long src_rows, long out_rows, int E, int N, int K) {
  const long far = (1l << 32) - (1 << 20);
  return E >= 1 && E <= MW_EXPERTS && K % MW_K == 0 && K >= 3 * MW_K && N % 8 == 0 &&
         ((down ? 1l : 2l) * N + MW_W) * K * 2 < far &&
         (down ? out_rows * N : src_rows * K) * 2 < far &&
         (long)MW_ROWS * N * 2 < far && (long)MW_ROWS * K * 2 < far &&
         out_rows < (1l << 30);
}

void moe_wide_launch(int down, void* out, const void* src, const void* w,
                     const int* rows, const float* s_w, const int* offs,
                     const int* counts, long src_rows, long out_rows, int E, int N,
                     int K, hipStream_t s) {
  if (out_rows == 0 || N == 0) return;
  const unsigned sb = (unsigned)(down ? 0 : src_rows * K * 2);
  const unsigned ob = (unsigned)(down ? out_rows * N * 2 : 0);
#define WIDE(D)                                                                \
  hipLaunchKernelGGL((moe_wide_kernel<D>), dim3(MW_CUS), dim3(256), 0, s,      \
                     (unsigned short*)out, (const unsigned short*)src,         \
                     (const unsigned short*)w, rows, s_w, offs, counts, E, N, K, \
                     sb, ob)
  if (down) WIDE(true);
  else WIDE(false);
#undef WIDE
}
