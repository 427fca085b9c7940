// Grouped MoE expert GEMMs for MI355X (gfx950): routing, expert sort, both
// expert products and the sum over a row's experts without a host readback.
//
// Two products over the expert-sorted assignment list:
//
//   moe_gate_up_silu: act[j, :] = silu(x[tok_j] @ Wg[e_j]^T) * (x[tok_j] @ Wu[e_j]^T)
//   moe_down_scale:   contrib[order[j], :] = (act[j] @ Wd[e_j]^T) * w_j
//
// GPT-OSS variants (per-expert biases + clamped swiglu, act_mode 1):
//   gate = min(g + bg, 7); up = clamp(u + bu, -7, 7)
//   act  = (up + 1) * gate * sigmoid(1.702 * gate)
//   contrib[order[j], :] = ((act[j] @ Wd[e_j]^T) + bd[e_j]) * w_j
// (matches models/llama.py MoEMLP._act_mul / the HF GptOss experts)
//
// Launch grids do not depend on the routing outcome: workgroups without a tile
// exit. Up to a few rows an expert both products come straight from memory, 16
// rows at a time (moe_few_kernel), bound by the weight stream (128 experts x 1536
// x 2048 at 64 rows: 133 us, 6 TB/s); moe_down_scale is its second one, if need be
// without a tile list. With more rows they run in 128 x 128 tiles (below), and
// whole prompts of many rows an expert in wider ones (moe_wide.hip).
#include "common.h"

#include <type_traits>

namespace {

constexpr int MOE_BN = 64;        // columns that moe_down_scale takes a multiple of
constexpr int MOE_THREADS = 256;  // 4 waves

typedef __attribute__((ext_vector_type(8))) short m_s16x8;

// ---------------------------------------------------------------------------
// Tile form. A tile is 128 rows of one expert x 128 weight rows (of gate and
// up: 64 each, 32 + 32 beside each other per wave, so that a lane holds a
// column's gate and up), four waves of 64 x 64 on mfma_f32_32x32x16_bf16, K in
// steps of 64 through LDS buffers that global_load_lds fills 16 bytes a lane,
// one barrier a step: two for the rows, which come out of the L2 a step ahead,
// three for the weights, which come out of memory two steps ahead (80 KB, two
// workgroups a CU). 16-byte chunks are XORed with (row >> 1): eight chunks a
// row, conflict-free over 16 rows of one chunk. Weights are the A operand: a
// lane ends with 4 neighbouring columns of a row, which go through the LDS to
// whole 16-byte stores.
// The tile list (moe_sort) holds only tiles that exist; workgroups are dealt to
// the XCDs in runs, and the tiles of an expert that share weight rows follow
// each other, so that these are read once into one L2 (tile by tile instead,
// 8 experts of 4096 x 14336 at 1024 rows each read 17 GB past the L2 and ran
// at 597 TFLOP/s). Halves of a wave's rows that an expert does not fill are
// not multiplied: three forms of the loop, without a branch inside, so that a
// 16-k's LDS reads fly under the products before it.
// The weights' first loads leave before the tile's rows are known, and what the
// end needs of the routing is read before the loop.
// Bound by the products and the weight stream alike: 254 rows per expert of
// 128 x (1536 + 768) x 2048 are 0.31 TFLOP and 1.2 GB a layer, 282 + 172 us (727
// and 596 TFLOP/s; with two buffers of each, branches between the products and
// the routing read at the end 312 + 198), 62 rows 155 + 96 (162 + 100), 4 rows
// 147 + 76 (150 + 76); 8 experts of 4096 x 14336 at 256 rows 636 + 407 (720 +
// 542). Tiles of 256 weight rows by eight waves, three buffers of each, one
// workgroup a CU: 278 to 286 + 176 to 179; of 256 in steps of 32: 291 to 312 +
// 181. Steps of 32 of 128 x 128 through three buffers: 322 to 330 + 187.
// ---------------------------------------------------------------------------
constexpr int MT_M = 128, MT_N = 128, MT_K = 64;
constexpr int MT_WB = 3;                     // weight buffers

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

DEVICE_INLINE unsigned int moe_pack(float lo, float hi) {
  const f32x2 v{lo, hi};
  return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2));
}

// FAR: rows of `src` lie further than 32 bits of bytes from its start.
template <bool DOWN, bool EXTM, bool FAR>
__global__ __launch_bounds__(MOE_THREADS, 2) void moe_tile_kernel(
    unsigned short* __restrict__ out,        // act [TK, I] | contrib [TK, H]
    const unsigned short* __restrict__ src,  // x [T, H] | act [TK, I]
    const unsigned short* __restrict__ w,    // [E, 2I, H] | [E, H, I]
    const int* __restrict__ rows,            // s_tok | order, [TK]
    const int* __restrict__ tiles,           // [max, 2] expert, first row
    const int* __restrict__ ntiles,          // [1]
    const int* __restrict__ offs, const int* __restrict__ counts,
    const float* __restrict__ flat_w,        // DOWN: [TK] routing weights
    const unsigned short* __restrict__ bias, // [E, 2I] | [E, H] or null
    int act_mode, int N, int K) {            // N = I | H
  constexpr int BUF = MT_M * MT_K;           // elements of a buffer
  static_assert(MT_M == MT_N, "rows and weights share their layout");
  // rows' buffers, then the weights'
  __shared__ __attribute__((aligned(16))) unsigned short lds[(2 + MT_WB) * BUF];
  constexpr int OW = DOWN ? MT_N : MT_N / 2; // columns of the result
  constexpr int NI = MT_M / 8 / 4;           // loads of a wave, 8 rows each

  const int nnt = N / OW;
  const int nwg = ntiles[0] * nnt;
  int wg = blockIdx.x;
  if (wg >= nwg) return;
  {
    const int q = nwg / 8, r = nwg % 8, xcd = wg % 8, idx = wg / 8;
    wg = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  // an expert's tiles take the same weight rows one after the other
  const int some = wg / nnt;                 // a tile of the same expert
  const int e = tiles[2 * some], cnt = counts[e];
  const int mt_n = (cnt + MT_M - 1) / MT_M;
  const int local = wg - (some - tiles[2 * some + 1] / MT_M) * nnt;
  const int nt = local / mt_n, m0 = local % mt_n * MT_M;
  const int first = offs[e] + m0;            // sorted row of the tile's first
  const int nrows = min(MT_M, cnt - m0);

  const int tid = threadIdx.x;
  const int lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int wm = wave >> 1, wn = wave & 1;
  const int lc = lane & 31, hf = lane >> 5;

  // A wave's load i brings rows (i * 4 + wave) * 8 .. of 128 bytes. Of gate and
  // up, 32 rows of one and 32 of the other take turns: a load is of one of them.
  const int nk = K / MT_K;
  const unsigned short* wbase =
      w + ((long)e * (DOWN ? N : 2 * N) + nt * OW) * K;
  unsigned int woff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    const int col = DOWN ? row : (row >> 6) * 32 + (row & 31);
    woff[i] = ((unsigned)col * K + chunk * 8) * 2;
  }
  auto load_weights = [&](int kt) {
    unsigned short* to = lds + (2 + kt % MT_WB) * BUF + wave * 8 * MT_K;
#pragma unroll
    for (int i = 0; i < NI; ++i)
      load_to_lds(wbase + (DOWN ? 0 : (long)(i & 1) * N * K) + kt * MT_K, woff[i],
               to + i * 32 * MT_K);
  };
  load_weights(0);
  const unsigned short* rbase = DOWN ? src + (long)first * K : src;
  std::conditional_t<FAR, unsigned long, unsigned int> roff[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int row = (i * 4 + wave) * 8 + lane / 8;
    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
    const int at = min(row, nrows - 1);
    roff[i] = DOWN ? at : rows[first + at];
    roff[i] = (roff[i] * K + chunk * 8) * 2;
  }
  auto load_rows = [&](int kt) {
    unsigned short* to = lds + (kt & 1) * BUF + wave * 8 * MT_K;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      if constexpr (FAR)
        load_to_lds(rbase + roff[i] / 2 + kt * MT_K, to + i * 32 * MT_K);
      else
        load_to_lds(rbase + kt * MT_K, roff[i], to + i * 32 * MT_K);
    }
  };
  // what the end needs of the routing
  constexpr int OC = OW / 8;                 // 16-byte chunks of a result row
  constexpr int NO = MT_M * OC / MOE_THREADS;
  int orow[NO];
  float rw[2] = {1.f, 1.f};
  if constexpr (DOWN) {
#pragma unroll
    for (int i = 0; i < NO; ++i)
      orow[i] = rows[first + min((tid + i * MOE_THREADS) / OC, nrows - 1)];
#pragma unroll
    for (int b = 0; b < 2; ++b)
      rw[b] = flat_w[rows[first + min(wm * 64 + b * 32 + lc, nrows - 1)]];
  }
  load_rows(0);
  if (nk > 1) load_weights(1);

  f32x16 acc[2][2];                          // [weight tile][row tile]
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  // NB: row tiles of this wave that hold rows
  auto products = [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    for (int kt = 0; kt < nk; ++kt) {
      // step kt is there: only the weights of the next were asked for later
      if (kt + 1 < nk)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NI) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (kt + 1 < nk) load_rows(kt + 1);
      if (kt + 2 < nk) load_weights(kt + 2);
      const unsigned short* rl = lds + (kt & 1) * BUF;
      const unsigned short* wl = lds + (2 + kt % MT_WB) * BUF;
      if constexpr (NB > 0) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int kk = 0; kk < MT_K / 16; ++kk) {
          u32x4 fw[2], fr[NB];
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const int at = wn * 64 + t * 32 + lc;
            fw[t] = *reinterpret_cast<const u32x4*>(
                wl + at * MT_K + ((kk * 2 + hf) ^ ((at >> 1) & 7)) * 8);
          }
#pragma unroll
          for (int t = 0; t < NB; ++t) {
            const int at = wm * 64 + t * 32 + lc;
            fr[t] = *reinterpret_cast<const u32x4*>(
                rl + at * MT_K + ((kk * 2 + hf) ^ ((at >> 1) & 7)) * 8);
          }
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int a = 0; a < 2; ++a)
              acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  __builtin_bit_cast(m_s16x8, fw[a]),
                  __builtin_bit_cast(m_s16x8, fr[b]), acc[a][b], 0, 0, 0);
        }
        __builtin_amdgcn_s_setprio(0);
      }
    }
  };
  const int mine = nrows - wm * 64;          // rows of this wave's half
  if (mine > 32) products(std::integral_constant<int, 2>{});
  else if (mine > 0) products(std::integral_constant<int, 1>{});
  else products(std::integral_constant<int, 0>{});
  __syncthreads();

  // acc[a][b][r]: weight row 8 (r>>2) + 4 hf + (r&3) of tile a, row lc of
  // tile b. Rows of the result through the LDS, 8-byte units XORed with row.
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int row = wm * 64 + b * 32 + lc;
#pragma unroll
    for (int a = 0; a < (DOWN ? 2 : 1); ++a)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int c = wn * (OW / 2) + a * 32 + rr * 8 + hf * 4;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = rr * 4 + j;
          if constexpr (DOWN) {
            float bd = 0.f;
            if constexpr (EXTM)
              if (bias != nullptr)
                bd = bf2f(bias[(long)e * N + nt * OW + c + j]);
            v[j] = (acc[a][b][r] + bd) * rw[b];
          } else {
            float g = acc[0][b][r], u = acc[1][b][r];
            if constexpr (EXTM) {
              if (bias != nullptr) {
                g += bf2f(bias[(long)e * 2 * N + nt * OW + c + j]);
                u += bf2f(bias[(long)e * 2 * N + N + nt * OW + c + j]);
              }
            }
            if (EXTM && act_mode == 1) {       // GPT-OSS clamped swiglu
              g = fminf(g, 7.f);
              u = fminf(fmaxf(u, -7.f), 7.f);
              v[j] = (u + 1.f) * g / (1.f + __expf(-1.702f * g));
            } else {
              v[j] = g / (1.f + __expf(-g)) * u;
            }
          }
        }
        *reinterpret_cast<u32x2*>(lds + row * OW + ((c / 4) ^ (row & 15)) * 4) =
            u32x2{moe_pack(v[0], v[1]), moe_pack(v[2], v[3])};
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NO; ++i) {
    const int u = tid + i * MOE_THREADS;
    const int row = u / OC, c = u % OC;
    if (row >= nrows) continue;
    const u32x2 a = *reinterpret_cast<const u32x2*>(
        lds + row * OW + ((2 * c) ^ (row & 15)) * 4);
    const u32x2 b = *reinterpret_cast<const u32x2*>(
        lds + row * OW + ((2 * c + 1) ^ (row & 15)) * 4);
    const long to = DOWN ? (long)orow[i] : (long)(first + row);
    *reinterpret_cast<u32x4*>(out + to * N + nt * OW + c * 8) =
        u32x4{a[0], a[1], b[0], b[1]};
  }
}

// Few rows an expert: 16 of them, 16 columns of gate and of up or 32 of the down product,
// straight from memory, k cut over the WAVES of a workgroup 64 by 64, DEPTH blocks of a
// wave in flight, sums through the LDS. More rows of an expert read its weights again.
// Bound by the weights: 128 experts of 768 x 2048 gate and up, 52 of them with rows, 56 us
// for tiles' 71, 126 133 for 142 (6 TB/s; at one row 8 experts, 96 tiles, 13.5 for 22).
// Three blocks in flight: four are more than 128 registers, and 175 us. Workgroups stay in
// the order of the experts over the XCDs: an expert's on one XCD, as the tiles are, gains
// 2 % where routing is even (130 us), but with half the rows at one expert takes 163 for
// 127. Waves and blocks by k so that few loads are past a wave's end: 8 waves of 1024 k,
// two blocks for three, 66 us for 4 waves' 48.
template <bool DOWN, int WAVES, int DEPTH>
__global__ __launch_bounds__(WAVES * WAVE_SIZE, 4) void moe_few_kernel(
    unsigned short* __restrict__ out,        // act [TK, I] | contrib [TK, H]
    const unsigned short* __restrict__ src,  // x [T, H] | act [TK, I]
    const unsigned short* __restrict__ w,    // [E, 2I, H] | [E, H, I]
    const int* __restrict__ rows,            // s_tok | order, [TK]
    const int* __restrict__ tiles,           // null: workgroups for every expert
    const int* __restrict__ ntiles,
    const int* __restrict__ offs, const int* __restrict__ counts,
    const float* __restrict__ flat_w,        // DOWN: [TK] routing weights
    const unsigned short* __restrict__ bias, // DOWN: [E, H] or null
    int N, int K) {                          // N = I | H
  constexpr int OW = DOWN ? 32 : 16;         // columns of the result
  constexpr int ST = 36;                     // floats of a row of sums
  __shared__ __attribute__((aligned(16))) float red[WAVES * 16 * ST];
  const int nnt = N / OW;
  const int wg = blockIdx.x, tile = wg / nnt;
  if (tiles != nullptr && tile >= ntiles[0]) return;
  const int e = tiles != nullptr ? tiles[2 * tile] : tile;
  const int r0 = tiles != nullptr ? tiles[2 * tile + 1] : 0;
  const int n0 = wg % nnt * OW;
  const int tid = threadIdx.x, lane = tid & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lc = lane & 15, lg = lane >> 4;
  const int nb = K / 64, n = wave < nb ? (nb - wave + WAVES - 1) / WAVES : 0;
  // rows lie a power of two apart: workgroups begin at places of their own
  const int rot = wg % nb;
  auto block = [&](int j) {
    const int i = min(wave + j * WAVES, nb - 1) + rot;
    return i < nb ? i : i - nb;
  };
  const char* wb[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
    wb[t] = (const char*)(w + (DOWN ? (long)e * N + n0 + t * 16
                                    : (long)e * 2 * N + t * N + n0) * K);
  const unsigned woff = ((unsigned)lc * K + lg * 8) * 2;
  const int first = offs[e];
  const int end = tiles != nullptr ? min(counts[e], r0 + MT_M) : counts[e];

  for (int m0 = r0; m0 < end; m0 += 16) {
    const int nrows = min(16, end - m0);
    const int at = min(lc, nrows - 1);
    const char* xb = (const char*)(DOWN ? src + (long)(first + m0) * K : src);
    const unsigned xoff =
        ((unsigned)(DOWN ? at : rows[first + m0 + at]) * K + lg * 8) * 2;
    u32x4 wr[DEPTH][2][2], xr[DEPTH][2];
    auto load = [&](int j, int in) {
      const long b = (long)block(j) * 128;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
          wr[in][t][c] = *reinterpret_cast<const u32x4*>(wb[t] + b + c * 64 + woff);
        xr[in][c] =
            *reinterpret_cast<const u32x4*>(xb + b + c * 64 + xoff);
      }
    };
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int j = 0; j < DEPTH; ++j) load(j, j);
    for (int q = 0; q < n; q += DEPTH) {
#pragma unroll
      for (int j = 0; j < DEPTH; ++j) {
        if (q + j < n) {
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int t = 0; t < 2; ++t)
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(m_s16x8, wr[j][t][c]),
                  __builtin_bit_cast(m_s16x8, xr[j][c]), acc[t], 0, 0, 0);
          if (q + j + DEPTH < n) load(q + j + DEPTH, j);
        }
      }
    }
    // column lg * 4 + r of row lc
    if (m0 > r0) __syncthreads();
#pragma unroll
    for (int t = 0; t < 2; ++t)
      *reinterpret_cast<f32x4*>(red + (wave * 16 + lc) * ST + t * 16 + lg * 4) = acc[t];
    __syncthreads();
    for (int u = tid; u < 16 * OW; u += WAVES * WAVE_SIZE) {
      const int row = u / OW, c = u % OW;
      if (row >= nrows) continue;
      float v[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < WAVES; ++i)
#pragma unroll
        for (int t = 0; t < (DOWN ? 1 : 2); ++t)
          v[t] += red[(i * 16 + row) * ST + t * 16 + c];
      if constexpr (DOWN) {
        const long to = rows[first + m0 + row];
        if (bias != nullptr) v[0] += bf2f(bias[(long)e * N + n0 + c]);
        out[to * N + n0 + c] = f2bf(v[0] * flat_w[to]);
      } else {
        out[(long)(first + m0 + row) * N + n0 + c] =
            f2bf(v[0] / (1.f + __expf(-v[0])) * v[1]);
      }
    }
  }
}

// Softmax routing: the k largest logits of a row in descending order (lowest
// index first among equals) and their weights: softmax over the chosen ones
// (renorm) or their share of the softmax over all. One wave per row, NV
// logits a lane, added up from `parts` here so that a product cut over k needs
// no launch to join it. A choice is a maximum over the wave without the LDS and a
// ballot for its place: value and place through the LDS, six exchanges of both for
// each of k, were most of the kernel (64 rows, 8 of 128 experts 8.2 us -> 4.4, 4188 rows
// 9.9 -> 6.2, 16384 23.8 -> 13.9). Bound by the launch and the latency of the logits.
template <int NV>
DEVICE_INLINE void moe_topk_row(int* experts, float* weights,
                                const float* logits, int lane, int E, int k,
                                int renorm, int parts = 1, long stride = 0) {
  float v[NV];
  unsigned taken = 0;
  bool nan = false;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int e = min(i * 64 + lane, E - 1);
    v[i] = logits[e];
  }
#pragma unroll 4
  for (int p = 1; p < parts; ++p)
#pragma unroll
    for (int i = 0; i < NV; ++i)
      v[i] += logits[p * stride + min(i * 64 + lane, E - 1)];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (i * 64 + lane >= E) {
      v[i] = -INFINITY;
      taken |= 1u << i;
    }
    nan |= v[i] != v[i];
  }
  const bool lost = __any(nan);        // one NaN is in every weight's sum
  float top = 0.f, mine = 0.f, sum = 0.f;
  int chosen = 0;
  for (int j = 0; j < k; ++j) {
    float best = -INFINITY;
#pragma unroll
    for (int i = 0; i < NV; ++i)
      best = fmaxf(best, taken >> i & 1 ? -INFINITY : v[i]);
    best = wave_reduce_max(best);
    int at = E - 1;                    // rows of NaN: any expert, in range
#pragma unroll
    for (int i = NV - 1; i >= 0; --i) {
      const unsigned long has = __ballot(!(taken >> i & 1) && v[i] == best);
      if (has != 0) at = i * 64 + __builtin_ctzl(has);
    }
    if ((at & 63) == lane) taken |= 1u << (at >> 6);
    if (j == 0) top = best;
    const float p = __expf(best - top);
    sum += p;
    if (lane == j) {
      mine = p;
      chosen = at;
    }
  }
  if (!renorm) {
    float all = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) all += __expf(v[i] - top);
    sum = wave_reduce_sum(all);
  }
  if (lane < k) {
    experts[lane] = chosen;
    weights[lane] = lost ? NAN : mine / sum;
  }
}

template <int NV>
__global__ __launch_bounds__(256) void moe_topk_kernel(
    int* __restrict__ experts,         // [T, k]
    float* __restrict__ weights,       // [T, k]
    const float* __restrict__ logits,  // [parts, T, E], to be added up
    int T, int E, int k, int renorm, int parts) {
  const int t = blockIdx.x * 4 + threadIdx.x / 64;
  if (t >= T) return;
  moe_topk_row<NV>(experts + (long)t * k, weights + (long)t * k,
                   logits + (long)t * E, threadIdx.x & 63, E, k, renorm, parts,
                   (long)T * E);
}

// The router's product and the choice in one launch, for bf16 rows and router
// weights of up to 16 experts: products of bf16 are exact in fp32, so bf16
// matrix instructions and their fp32 sums stand for the fp32 product of the
// casted operands. A workgroup takes 16 rows, its 16 waves the 128-k blocks in
// turn; the sums meet in the LDS, where each wave then chooses for one row.
// Bound by latency: 9 us at 64 rows over 8 experts of 4096, 12 at 4068 (cast,
// fp32 product and choice apart: 15 and 40). With more experts the router's
// weights, read again by every workgroup, take over (128 of 2048 at 64 rows
// 25): those take the tiled product's parts and the choice above.
__global__ __launch_bounds__(1024) void moe_route_kernel(
    int* __restrict__ experts,               // [T, k]
    float* __restrict__ weights,             // [T, k]
    const unsigned short* __restrict__ x,    // [T, H]
    const unsigned short* __restrict__ w,    // [E, H]
    int T, int E, int H, int k, int renorm) {
  __shared__ float red[16 * 16 * 16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE_SIZE);
  const int lc = lane & 15, lg = lane >> 4;
  const int t0 = blockIdx.x * 16;
  const unsigned short* xp = x + (long)min(t0 + lc, T - 1) * H + lg * 8;
  const unsigned short* wp = w + (long)min(lc, E - 1) * H + lg * 8;
  f32x4 acc{0.f, 0.f, 0.f, 0.f};
  for (int b = wave; b < H / 128; b += 16)
#pragma unroll
    for (int c = 0; c < 4; ++c)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(m_s16x8, *reinterpret_cast<const u32x4*>(
                                          xp + b * 128 + c * 32)),
          __builtin_bit_cast(m_s16x8, *reinterpret_cast<const u32x4*>(
                                          wp + b * 128 + c * 32)),
          acc, 0, 0, 0);
  // D[row = lg*4 + r][expert = lc]
#pragma unroll
  for (int r = 0; r < 4; ++r)
    red[(wave * 16 + lg * 4 + r) * 16 + lc] = acc[r];
  __syncthreads();
  if (tid < 256) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) v += red[i * 256 + tid];
    red[tid] = v;                            // read by this thread alone so far
  }
  __syncthreads();
  if (t0 + wave < T)
    moe_topk_row<1>(experts + (long)(t0 + wave) * k,
                    weights + (long)(t0 + wave) * k, red + wave * 16, lane, E,
                    k, renorm);
}

constexpr int MOE_MAX_E = 4096;

// Counting sort of the assignments by expert: counts, offsets, the sorted rows,
// their weights where these are given, and the tile list. The order within an expert is free: a row's result does
// not depend on its place. A short list is one workgroup's (about 5 us at 512
// assignments; a radix sort, a scatter and the casts around them took 100).
// Longer ones (32544 took it 37 us) are cut into slices of MOE_SLICE: a first
// kernel counts each slice's experts, and every workgroup of the second adds
// up for itself where its slice begins in each expert (eight slices' counts at a time:
// 33504 assignments to 128 experts 13.4 us -> 10.4, one by one to now).
constexpr int MOE_SLICE = 2048;

template <typename F>
DEVICE_INLINE void moe_walk(const int* experts, int from, int to, int E, F f) {
  int i = from + (int)threadIdx.x;
  for (; i + 7 * 1024 < to; i += 8 * 1024) {  // eight loads in flight a thread
    int e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = experts[i + j * 1024];
#pragma unroll
    for (int j = 0; j < 8; ++j) f(i + j * 1024, min(max(e[j], 0), E - 1));
  }
  for (; i < to; i += 1024) f(i, min(max(experts[i], 0), E - 1));
}

__global__ __launch_bounds__(1024) void moe_count_kernel(
    int* __restrict__ hist,            // [slices, E]
    const int* __restrict__ experts, int TK, int E) {
  __shared__ int cnt[MOE_MAX_E];
  for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
  __syncthreads();
  const int from = blockIdx.x * MOE_SLICE;
  moe_walk(experts, from, min(TK, from + MOE_SLICE), E,
           [&](int, int e) { atomicAdd(&cnt[e], 1); });
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += 1024)
    hist[(long)blockIdx.x * E + e] = cnt[e];
}

// From a thread's counts of its experts (ept of them from tid * ept on) to their offsets
// and the tile list, and to the next free place of each expert's in `cnt`, `before`
// places in where others come first. By a whole workgroup of 1024; no barrier behind.
template <int EPT>
DEVICE_INLINE void moe_offsets(int* cnt, const int (&c)[EPT], const int (&before)[EPT],
                               int ept, bool lead, int* counts, int* offs, int* tiles,
                               int* ntiles, int E) {
  __shared__ int wsum[2][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int a = 0, b = 0;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    a += c[j];
    b += (c[j] + MT_M - 1) / MT_M;
  }
  const int own_a = a, own_b = b;
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {   // inclusive sums over the wave
    const int x = __shfl_up(a, m, 64), y = __shfl_up(b, m, 64);
    if (lane >= m) {
      a += x;
      b += y;
    }
  }
  if (lane == 63) {
    wsum[0][wave] = a;
    wsum[1][wave] = b;
  }
  __syncthreads();
  for (int i = 0; i < wave; ++i) {
    a += wsum[0][i];
    b += wsum[1][i];
  }
  if (lead && tid == 1023) ntiles[0] = b;
  a -= own_a;
  b -= own_b;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid * ept + j;
    if (j >= ept || e >= E) continue;
    cnt[e] = a + before[j];
    if (lead) {
      counts[e] = c[j];
      offs[e] = a;
      for (int r = 0; r < c[j]; r += MT_M, ++b) {
        tiles[2 * b] = e;
        tiles[2 * b + 1] = r;
      }
    }
    a += c[j];
  }
}

// gridDim.x slices with their counts in `hist`, or one workgroup without.
__global__ __launch_bounds__(1024) void moe_sort_kernel(
    int* __restrict__ order, int* __restrict__ s_tok,  // [TK]
    float* __restrict__ s_w, const float* __restrict__ flat_w,  // [TK] or null
    int* __restrict__ counts, int* __restrict__ offs,  // [E]
    int* __restrict__ tiles, int* __restrict__ ntiles,
    const int* __restrict__ experts, const int* __restrict__ hist, int TK,
    int E, int k) {
  __shared__ int cnt[MOE_MAX_E];       // counts, then the next free places
  constexpr int EPT = MOE_MAX_E / 1024;
  const int tid = threadIdx.x;
  const int from = hist != nullptr ? blockIdx.x * MOE_SLICE : 0;
  const int to = hist != nullptr ? min(TK, from + MOE_SLICE) : TK;
  // thread tid owns experts EPT * tid .. (one each up to 1024 of them)
  const int ept = E <= 1024 ? 1 : EPT;
  int c[EPT], before[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) c[j] = before[j] = 0;
  if (hist == nullptr) {
    for (int e = tid; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
    moe_walk(experts, from, to, E, [&](int, int e) { atomicAdd(&cnt[e], 1); });
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = tid * ept + j;
    if (j >= ept || e >= E) continue;
    if (hist == nullptr) {
      c[j] = cnt[e];
    } else {
      const int slices = gridDim.x;
      for (int b0 = 0; b0 < slices; b0 += 8) {   // eight loads in flight
        int v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i)
          v[i] = hist[(long)min(b0 + i, slices - 1) * E + e];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if (b0 + i < slices) c[j] += v[i];
          if (b0 + i < (int)blockIdx.x) before[j] += v[i];
        }
      }
    }
  }
  moe_offsets(cnt, c, before, ept, blockIdx.x == 0, counts, offs, tiles, ntiles, E);
  __syncthreads();
  moe_walk(experts, from, to, E, [&](int i, int e) {
    const int at = atomicAdd(&cnt[e], 1);
    order[at] = i;
    s_tok[at] = i / k;
    if (s_w != nullptr) s_w[at] = flat_w[i];
  });
}

// moe_topk_kernel and moe_sort_kernel in one launch, for up to a row a wave of one
// workgroup, which counts in the LDS as it chooses and goes on with what it chose. Bound
// by its chain and, from 8 waves on, by their instructions on one CU: us, two launches /
// one at 1 / 8 / 16 rows, 8 of 128 experts 6.3 / 5.2, 7.1 / 5.7, 7.0 / 7.0, 6 of 64 5.8 /
// 4.6, 6.3 / 4.9, 6.4 / 5.7, 8 of 256 6.9 / 6.5, 7.4 / 7.1, 7.5 / 8.6; two rows a wave
// 7.3 / 10.4 and more.
constexpr int MOE_CHOOSE = 16;

template <int NV>
__global__ __launch_bounds__(1024) void moe_choose_kernel(
    int* __restrict__ experts, float* __restrict__ weights,  // [T, k]
    int* __restrict__ order, int* __restrict__ s_tok,        // [T * k]
    int* __restrict__ counts, int* __restrict__ offs,        // [E]
    int* __restrict__ tiles, int* __restrict__ ntiles,
    const float* __restrict__ logits,  // [parts, T, E], to be added up
    int T, int E, int k, int renorm, int parts) {
  __shared__ int cnt[NV * 64];
  __shared__ int chosen[MOE_CHOOSE * 64];
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < E) cnt[tid] = 0;
  __syncthreads();
  const int t = tid >> 6;
  if (t < T) {
    moe_topk_row<NV>(chosen + t * k, weights + (long)t * k, logits + (long)t * E, lane,
                     E, k, renorm, parts, (long)T * E);
    if (lane < k) atomicAdd(&cnt[chosen[t * k + lane]], 1);
  }
  __syncthreads();
  const int c[1] = {tid < E ? cnt[tid] : 0}, before[1] = {0};
  moe_offsets(cnt, c, before, 1, true, counts, offs, tiles, ntiles, E);
  __syncthreads();
  for (int i = tid; i < T * k; i += 1024) {
    const int e = chosen[i], at = atomicAdd(&cnt[e], 1);
    experts[i] = e;
    order[at] = i;
    s_tok[at] = i / k;
  }
}

// The tile list alone, from counts that the caller brings.
__global__ __launch_bounds__(64) void moe_tiles_kernel(
    int* __restrict__ tiles, int* __restrict__ ntiles,
    const int* __restrict__ counts, int E, int max_tiles) {
  if (threadIdx.x != 0) return;
  int n = 0;
  for (int e = 0; e < E; ++e)
    for (int r = 0; r < counts[e] && n < max_tiles; r += MT_M, ++n) {
      tiles[2 * n] = e;
      tiles[2 * n + 1] = r;
    }
  ntiles[0] = n;
}

// out[t] = sum over the k contributions of row t, in fp32 in their order.
// Bound by reading them once.
__global__ __launch_bounds__(256) void moe_sum_kernel(
    unsigned short* __restrict__ out,            // [T, H]
    const unsigned short* __restrict__ contrib,  // [T, k, H]
    long units, int k, int H) {
  const int hu = H / 8;
  for (long u = (long)blockIdx.x * 256 + threadIdx.x; u < units;
       u += (long)gridDim.x * 256) {
    const unsigned short* p = contrib + (u / hu) * k * H + (u % hu) * 8;
    float s[8];
    bf8_to_f32(*reinterpret_cast<const u16x8*>(p), s);
    for (int j = 1; j < k; ++j) {
      float f[8];
      bf8_to_f32(*reinterpret_cast<const u16x8*>(p + (long)j * H), f);
#pragma unroll
      for (int i = 0; i < 8; ++i) s[i] += f[i];
    }
    *reinterpret_cast<u32x4*>(out + u * 8) =
        u32x4{moe_pack(s[0], s[1]), moe_pack(s[2], s[3]),
              moe_pack(s[4], s[5]), moe_pack(s[6], s[7])};
  }
}

}  // namespace

void moe_topk_launch(int* experts, float* weights, const float* logits, int T,
                     int E, int k, int renorm, int parts,
                     int* err_unsupported, hipStream_t s) {
  *err_unsupported = 0;
  if (E < 1 || E > 1024 || k < 1 || k > 64 || k > E) {
    *err_unsupported = 1;
    return;
  }
  if (T == 0) return;
#define TOPK(NV)                                                             \
  hipLaunchKernelGGL((moe_topk_kernel<NV>), dim3((T + 3) / 4), dim3(256), 0, \
                     s, experts, weights, logits, T, E, k, renorm, parts)
  if (E <= 64) TOPK(1);
  else if (E <= 128) TOPK(2);
  else if (E <= 256) TOPK(4);
  else if (E <= 512) TOPK(8);
  else TOPK(16);
#undef TOPK
}

// logits [parts, T, E]; tiles of T * k / 128 + E pairs
void moe_choose_launch(int* experts, float* weights, int* order, int* s_tok, int* counts,
                       int* offs, int* tiles, int* ntiles, const float* logits, int T,
                       int E, int k, int renorm, int parts, int* err_unsupported,
                       hipStream_t s) {
  *err_unsupported = E < 1 || E > 256 || k < 1 || k > 64 || k > E || T < 1 ||
                     T > MOE_CHOOSE;
  if (*err_unsupported) return;
#define CHOOSE(NV)                                                                 \
  hipLaunchKernelGGL((moe_choose_kernel<NV>), dim3(1), dim3(1024), 0, s, experts,  \
                     weights, order, s_tok, counts, offs, tiles, ntiles, logits, T, \
                     E, k, renorm, parts)
  if (E <= 64) CHOOSE(1);
  else if (E <= 128) CHOOSE(2);
  else CHOOSE(4);
#undef CHOOSE
}

void moe_route_launch(int* experts, float* weights, const void* x,
                      const void* w, int T, int E, int H, int k, int renorm,
                      int* err_unsupported, hipStream_t s) {
  *err_unsupported = E < 1 || E > 16 || k < 1 || k > E || H < 128 ||
                     H % 128 != 0;
  if (*err_unsupported || T == 0) return;
  hipLaunchKernelGGL(moe_route_kernel, dim3((T + 15) / 16), dim3(1024), 0, s,
                     experts, weights, (const unsigned short*)x,
                     (const unsigned short*)w, T, E, H, k, renorm);
}

// hist: [slices, E] for moe_sort_slices(TK) > 0 of them, else unused
int moe_sort_slices(int TK) {
  return TK > 2 * MOE_SLICE ? (TK + MOE_SLICE - 1) / MOE_SLICE : 0;
}

void moe_sort_launch(int* order, int* s_tok, float* s_w, const float* flat_w,
                     int* counts, int* offs, int* tiles, int* ntiles, int* hist,
                     const int* experts, int TK, int E, int k,
                     int* err_unsupported, hipStream_t s) {
  *err_unsupported = E < 1 || E > MOE_MAX_E;
  if (*err_unsupported) return;
  const int slices = moe_sort_slices(TK);
  if (slices > 0)
    hipLaunchKernelGGL(moe_count_kernel, dim3(slices), dim3(1024), 0, s, hist,
                       experts, TK, E);
  hipLaunchKernelGGL(moe_sort_kernel, dim3(slices > 0 ? slices : 1),
                     dim3(1024), 0, s, order, s_tok, s_w, flat_w, counts, offs,
                     tiles, ntiles, experts, slices > 0 ? hist : nullptr, TK, E, k);
}

void moe_tiles_launch(int* tiles, int* ntiles, const int* counts, int E,
                      int max_tiles, hipStream_t s) {
  hipLaunchKernelGGL(moe_tiles_kernel, dim3(1), dim3(64), 0, s, tiles, ntiles,
                     counts, E, max_tiles);
}

void moe_sum_launch(void* out, const void* contrib, long T, int k, int H,
                    hipStream_t s) {
  const long units = T * (H / 8);
  if (units == 0) return;
  const long grid = (units + 255) / 256;
  hipLaunchKernelGGL(moe_sum_kernel, dim3(grid > 8192 ? 8192 : (int)grid),
                     dim3(256), 0, s, (unsigned short*)out,
                     (const unsigned short*)contrib, units, k, H);
}

// max_tiles bounds the tile list: no more than TK / 128 + E tiles exist.
void moe_tile_launch(int down, void* out, const void* src, const void* w,
                     const int* rows, const int* tiles, const int* ntiles,
                     const int* offs, const int* counts, const float* flat_w,
                     const void* bias, int act_mode, long src_rows,
                     int max_tiles, int N, int K, int* err_unsupported,
                     hipStream_t s) {
  const int ow = down ? MT_N : MT_N / 2;
  *err_unsupported = N % ow != 0 || K % MT_K != 0;
  if (*err_unsupported || max_tiles == 0) return;
  const bool extm = bias != nullptr || act_mode != 0;
  const bool far = !down && src_rows * K * 2 >= 1l << 32;
#define TILE(D, X, F)                                                         \
  hipLaunchKernelGGL((moe_tile_kernel<D, X, F>),                              \
                     dim3((unsigned)max_tiles * (N / ow)), dim3(MOE_THREADS), \
                     0, s, (unsigned short*)out, (const unsigned short*)src,  \
                     (const unsigned short*)w, rows, tiles, ntiles, offs,     \
                     counts, flat_w, (const unsigned short*)bias, act_mode,   \
                     N, K)
  if (down) {
    if (extm) TILE(true, true, false);
    else TILE(true, false, false);
  } else if (far) {
    if (extm) TILE(false, true, true);
    else TILE(false, false, true);
  } else {
    if (extm) TILE(false, true, false);
    else TILE(false, false, false);
  }
#undef TILE
}

// Without tiles every expert has workgroups, of which those without rows exit.
static void moe_few(int down, void* out, const void* src, const void* w,
                    const int* rows, const int* tiles, const int* ntiles,
                    const int* offs, const int* counts, const float* flat_w,
                    const void* bias, long groups, int N, int K, hipStream_t s) {
#define FEW(D, W, B)                                                            \
  hipLaunchKernelGGL((moe_few_kernel<D, W, B>),                                 \
                     dim3((unsigned)groups * (N / (D ? 32 : 16))),              \
                     dim3(W * WAVE_SIZE), 0, s, (unsigned short*)out,           \
                     (const unsigned short*)src, (const unsigned short*)w,      \
                     rows, tiles, ntiles, offs, counts, flat_w,                 \
                     (const unsigned short*)bias, N, K)
#define FEW_K(D)                           \
  do {                                     \
    if (K >= 1536) FEW(D, 8, 3);           \
    else if (K > 512) FEW(D, 4, 3);        \
    else FEW(D, 4, 2);                     \
  } while (0)
  if (down) FEW_K(true);
  else FEW_K(false);
#undef FEW_K
#undef FEW
}

// tiles of moe_sort's list: one an expert of those that have rows, and one for 128 rows
void moe_few_launch(int down, void* out, const void* src, const void* w,
                    const int* rows, const int* tiles, const int* ntiles,
                    const int* offs, const int* counts, const float* flat_w,
                    long src_rows, long TK, int E, int N, int K,
                    int* err_unsupported, hipStream_t s) {
  const int ow = down ? 32 : 16;
  const long groups = (TK < E ? TK : E) + TK / MT_M;
  *err_unsupported = N % ow != 0 || K % 64 != 0 || K == 0 ||
                     groups * (N / ow) >= 1l << 31 ||
                     (!down && src_rows * K * 2 >= 1l << 32);
  if (*err_unsupported || groups == 0 || N == 0) return;
  moe_few(down, out, src, w, rows, tiles, ntiles, offs, counts, flat_w, nullptr,
          groups, N, K, s);
}

void moe_down_scale_launch(void* contrib, const void* act, const void* w,
                           const int* offs, const int* counts,
                           const int* order, const float* flat_w,
                           const void* bias, const int* tiles, const int* ntiles,
                           long TK, int E,
                           int H, int I, int* err_unsupported, hipStream_t s) {
  *err_unsupported = H % MOE_BN != 0 || I % 128 != 0 || I == 0;
  const long groups = tiles != nullptr ? (TK < E ? TK : E) + TK / MT_M : E;
  if (*err_unsupported || groups == 0 || H == 0) return;
  moe_few(1, contrib, act, w, order, tiles, ntiles, offs, counts, flat_w, bias,
          groups, H, I, s);
}
