// Causal flash attention of prompt rows for MI355X (gfx950) on MFMA: whole
// prompts (keys and values in the step's own rows) and rows behind a cached
// history (keys and values in the paged pool): flash_prefill_kernel for all head
// sizes and options, flash_rows_kernel for heads of 128 channels without options.
//
// Replaces the prefill attention the reference gets from vLLM/SGLang.
//
// Of the first:
//  - a workgroup owns 128 query rows of one head, 4 waves x 32 rows, and
//    walks the keys 64 at a time; mfma_f32_32x32x16_bf16, lane layouts
//      A: lane holds A[row = l&31][k = (l>>5)*8 + j]
//      B: lane holds B[k = (l>>5)*8 + j][col = l&31]
//      D: lane holds D[row = 8*(r>>2) + 4*(l>>5) + (r&3)][col = l&31]
//    (twice the work per LDS byte of the 16x16x32 form).
//  - S^T = K Q^T, so a lane holds 32 scores of ONE query row: maximum and sum
//    are in-lane but for one exchange with lane^32, and the rescaling factor
//    of a row sits in the lanes that hold the row's output.
//  - O^T = V^T P^T takes P as it lies in the registers: the k slots of a
//    product are the keys {4h..4h+3, 8+4h..8+4h+3} of 16 (h = l>>5), and V^T
//    is read in the same order (two 8-byte LDS reads).
//  - V is transposed on its way into the LDS: a thread loads 4 rows x 8
//    channels with 16-byte loads, pairs the rows with v_perm and writes eight
//    4-key units. VT rows have 68 elements and units are XORed with
//    2 * (d/32): conflict-free writes (32 lanes, 4 x 8-aligned windows) and
//    reads (17 d mod 32). K rows keep their order, 16-byte chunks XORed with
//    the row.
//  - two LDS buffers: the next tile's global loads fly under this tile's
//    products, one barrier per tile; 66 KB, two workgroups a CU, so one's
//    exponentials run beside the other's products.
//  - the running maximum moves only when a row's scores pass it by 2^8: P is
//    then at most 2^8, which neither bf16 P nor the fp32 sums notice, and the
//    output is rescaled in few tiles.
//  - workgroups of one kv head go to one XCD (head order below), whose L2
//    then holds that head's keys and values; the tiles with the most keys
//    start first.
//
// Bound by the products and exponentials together (16 + 16 MFMAs of 32 cycles
// and 32 exponentials of 16 cycles a wave and tile).
#include "common.h"

namespace {

constexpr int BQ = 128;
constexpr int BK = 64;
constexpr int PF_WAVES = 4;
constexpr int PF_THREADS = PF_WAVES * WAVE_SIZE;
constexpr int VT_ROW = BK + 4;     // elements of a V^T row in the LDS
constexpr int PP_BS = 16;          // pool block size (tokens per KV block)
constexpr float LOG2E = 1.4426950408889634f;
constexpr float SLACK = 8.f;       // see "running maximum" above

typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

DEVICE_INLINE f32x4 mfma16x16x32_bf16(u16x8 a, u16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(s16x8, a), __builtin_bit_cast(s16x8, b), c, 0, 0, 0);
}

DEVICE_INLINE f32x16 mfma32x32x16_bf16(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(
      __builtin_bit_cast(s16x8, a), __builtin_bit_cast(s16x8, b), c, 0, 0, 0);
}

DEVICE_INLINE unsigned int pack_bf16(float lo, float hi) {
  const f32x2 v{lo, hi};
  return __builtin_bit_cast(unsigned int,
                            __builtin_convertvector(v, bf16x2));
}

// A wave's 32 rows of the result (o: channels 32 n + 8 rr + 4 (l>>5) .. of row
// l & 31) through its own part of the LDS to whole rows: unit u (4 channels) of
// row r at u ^ (r & 15).
template <int DVK>
DEVICE_INLINE void store_rows(unsigned short* __restrict__ out,
                              unsigned short* ol, const f32x16 (&o)[DVK / 32],
                              float inv, int row0, int first, int nnew, int Hq,
                              int qh, int lane) {
  constexpr int OC = DVK / 8;              // 16-byte chunks of an output row
  const int lc = lane & 31, hf = lane >> 5;
#pragma unroll
  for (int n = 0; n < DVK / 32; ++n)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      u32x2 w;
      w[0] = pack_bf16(o[n][rr * 4] * inv, o[n][rr * 4 + 1] * inv);
      w[1] = pack_bf16(o[n][rr * 4 + 2] * inv, o[n][rr * 4 + 3] * inv);
      const int unit = n * 8 + rr * 2 + hf;
      *reinterpret_cast<u32x2*>(ol + lc * DVK + (unit ^ (lc & 15)) * 4) = w;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < OC / 2; ++i) {
    const int u = lane + i * WAVE_SIZE;
    const int r = u / OC, c = u % OC;
    const u32x2 a = *reinterpret_cast<const u32x2*>(
        ol + r * DVK + ((2 * c) ^ (r & 15)) * 4);
    const u32x2 b = *reinterpret_cast<const u32x2*>(
        ol + r * DVK + ((2 * c + 1) ^ (r & 15)) * 4);
    if (first + r < nnew)
      *reinterpret_cast<u32x4*>(
          out + ((long)(row0 + first + r) * Hq + qh) * DVK + c * 8) =
          u32x4{a[0], a[1], b[0], b[1]};
  }
}

// EXT: 1 sinks / sliding window, 2 softcap (and those). Forms of their own,
// because a short prompt is one pass over the code (77 rows of 64 heads of 64
// on 8, us: 7.3, 8.4 and 11.4; with all of it in one kernel 8.9, 8.9 and 14.6).
// PAGED: k / v are pools [nblocks, Hkv, 16, D]; otherwise rows of the batch.
// A tile: the sequence's first row in q and out, the tile's first row within
// the sequence's rows, the cached tokens in front of them, their number, and
// the sequence's row of the block tables.
template <int D, int DVK, int EXT, bool PAGED>
__global__ __launch_bounds__(PF_THREADS, D > 128 ? 1 : 2)
void flash_prefill_kernel(
    unsigned short* __restrict__ out,      // [T, Hq, DVK]
    const unsigned short* __restrict__ q,  // [T, Hq, D]
    const unsigned short* __restrict__ k,
    const unsigned short* __restrict__ v,
    const int* __restrict__ block_tables,  // [nseq, maxb]
    const int* __restrict__ tile_start, const int* __restrict__ tile_q0,
    const int* __restrict__ tile_hist, const int* __restrict__ tile_new,
    const int* __restrict__ tile_seq,
    int Hq, int Hkv, int maxb, float scale,
    long qs, long ks, long vs,             // row strides (elements)
    const float* __restrict__ sinks,       // [Hq] or null
    int window,                            // 0 = full causal
    float softcap) {                       // 0 = off (Gemma-2 tanh cap)
  constexpr int CH = D / 8;                // 16-byte chunks of a key row
  constexpr int KU = CH / 4;               // K chunks a lane stages
  constexpr int VB = (DVK / 8 * 4 + 63) / 64;  // V blocks a lane stages
  constexpr int KMASK = D % 128 == 0 ? 15 : 7;
  constexpr int QK = D / 16;
  constexpr int NT = DVK / 32;
  constexpr int K_ELEMS = BK * D;
  constexpr int BUF = K_ELEMS + DVK * VT_ROW;

  static_assert(2 * BUF >= BQ * DVK, "the output goes through the buffers");
  __shared__ __attribute__((aligned(16))) unsigned short lds[2 * BUF];

  // heads of one kv head on one XCD (workgroups go round the 8 XCDs)
  int qh = blockIdx.x % Hq;
  if (Hq % 8 == 0) qh = (qh % 8) * (Hq / 8) + qh / 8;
  const int tile = (gridDim.x - 1 - blockIdx.x) / Hq;
  const int kvh = qh / (Hq / Hkv);
  const int row0 = tile_start[tile];
  const int q0 = tile_q0[tile];
  if (q0 % BQ != 0) return;          // the second half of a list of 64-row tiles
  const int hist = PAGED ? tile_hist[tile] : 0;
  const int nnew = tile_new[tile];
  const int len = hist + nnew;
  const int* bt = PAGED ? block_tables + (long)tile_seq[tile] * maxb : nullptr;

  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lc = lane & 31;
  const int hf = lane >> 5;
  // The lane's own part of every LDS and memory address does not change from
  // tile to tile; at 256 channels keeping all of them took more than 512
  // registers (284 bytes a lane in scratch, 77 rows 18.8 us; worked out anew in
  // each tile 13.7, and 2000 rows 191 -> 126).
  auto lane_again = [&] {
    int l = lane;
    if constexpr (D > 192) asm volatile("" : "+v"(l));
    return l;
  };

  // this wave's 32 query rows as the B operand
  const int qrow = q0 + wave * 32 + lc;            // within the new rows
  const int qpos = hist + qrow;
  u32x4 qf[QK];
  {
    const unsigned short* qp =
        q + (long)(row0 + min(qrow, nnew - 1)) * qs + (long)qh * D + hf * 8;
#pragma unroll
    for (int kk = 0; kk < QK; ++kk)
      qf[kk] = *reinterpret_cast<const u32x4*>(qp + kk * 16);
  }

  float m = -INFINITY, l = 0.f;
  f32x16 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  const int lo_wave = hist + q0 + wave * 32;       // this wave's first row
  const int kv_end = min(len, hist + q0 + BQ);     // causal bound
  const int kt_end = (kv_end + BK - 1) / BK;
  // the first tile any row of the workgroup can see
  int kt0 = 0;
  if constexpr (EXT > 0)
    if (window > 0) kt0 = max(0, hist + q0 - window + 1) / BK;

  u32x4 kst[KU], vst[VB][4];

  // wave w stages rows 16 w .. 16 w + 15 of a tile (one page of a pool)
  auto issue = [&](int kt) {
    const int lane = lane_again();
    const int kv0 = kt * BK + wave * 16;
    const unsigned short *kp, *vp;
    long kstep, vstep;
    int last;                                      // rows behind it repeat it
    if constexpr (PAGED) {
      const int page = min(kv0, len - 1) / PP_BS;
      const long at = ((long)bt[page] * Hkv + kvh) * PP_BS;
      kp = k + at * D;
      vp = v + at * DVK;
      kstep = D;
      vstep = DVK;
      last = PP_BS - 1;
    } else {
      const int r = min(kv0, len - 1);
      kp = k + (long)(row0 + r) * ks + (long)kvh * D;
      vp = v + (long)(row0 + r) * vs + (long)kvh * DVK;
      kstep = ks;
      vstep = vs;
      last = min(15, len - 1 - r);
    }
#pragma unroll
    for (int i = 0; i < KU; ++i) {
      const int u = lane + i * WAVE_SIZE;
      kst[i] = *reinterpret_cast<const u32x4*>(
          kp + min(u / CH, last) * kstep + (u % CH) * 8);
    }
#pragma unroll
    for (int b = 0; b < VB; ++b) {
      const int u = lane + b * WAVE_SIZE;
      if (DVK >= 128 || u < DVK / 2) {
        const int r0 = u / (DVK / 8) * 4, d0 = u % (DVK / 8) * 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          vst[b][j] = *reinterpret_cast<const u32x4*>(
              vp + min(r0 + j, last) * vstep + d0);
          // a page's rows behind the sequence's end are not the sequence's
          if (PAGED && kv0 + r0 + j >= len) vst[b][j] = u32x4{0, 0, 0, 0};
        }
      }
    }
  };

  auto stash = [&](unsigned short* buf) {
    const int lane = lane_again();
    unsigned short* vt = buf + K_ELEMS;
#pragma unroll
    for (int i = 0; i < KU; ++i) {
      const int u = lane + i * WAVE_SIZE;
      const int row = wave * 16 + u / CH;
      *reinterpret_cast<u32x4*>(
          buf + row * D + (((u % CH) ^ (row & KMASK)) * 8)) = kst[i];
    }
#pragma unroll
    for (int b = 0; b < VB; ++b) {
      const int u = lane + b * WAVE_SIZE;
      if (DVK >= 128 || u < DVK / 2) {
        const int unit = wave * 4 + u / (DVK / 8), d0 = u % (DVK / 8) * 8;
        unsigned short* at =
            vt + d0 * VT_ROW + (unit ^ (2 * ((d0 >> 5) & 3))) * 4;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          // channels 2w and 2w + 1 of four rows
          u32x2 e, f;
          e[0] = __builtin_amdgcn_perm(vst[b][1][w], vst[b][0][w], 0x05040100u);
          e[1] = __builtin_amdgcn_perm(vst[b][3][w], vst[b][2][w], 0x05040100u);
          f[0] = __builtin_amdgcn_perm(vst[b][1][w], vst[b][0][w], 0x07060302u);
          f[1] = __builtin_amdgcn_perm(vst[b][3][w], vst[b][2][w], 0x07060302u);
          *reinterpret_cast<u32x2*>(at + (2 * w) * VT_ROW) = e;
          *reinterpret_cast<u32x2*>(at + (2 * w + 1) * VT_ROW) = f;
        }
      }
    }
  };

  const float sc = EXT == 2 ? scale / softcap : scale * LOG2E;
  issue(kt0);
  stash(lds);
  __syncthreads();
  for (int kt = kt0; kt < kt_end; ++kt) {
    const int kv0 = kt * BK;
    const unsigned short* kl = lds + ((kt - kt0) & 1) * BUF;
    const unsigned short* vt = kl + K_ELEMS;
    const bool more = kt + 1 < kt_end;
    if (more) issue(kt + 1);

    bool live = kv0 <= lo_wave + 31;               // not above the diagonal
    if constexpr (EXT > 0)
      live = live && !(window > 0 && kv0 + BK <= lo_wave - window + 1);
    if (live) {
      const int la = lane_again(), lc = la & 31, hf = la >> 5;
      f32x16 st[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) st[t][r] = 0.f;
        const int row = t * 32 + lc;
#pragma unroll
        for (int kk = 0; kk < QK; ++kk) {
          const u32x4 a = *reinterpret_cast<const u32x4*>(
              kl + row * D + (((kk * 2 + hf) ^ (row & KMASK)) * 8));
          st[t] = mfma32x32x16_bf16(a, qf[kk], st[t]);
        }
      }
      // scores in powers of two
      bool edge = kv0 + BK - 1 > lo_wave || kv0 + BK > len;
      if constexpr (EXT > 0) edge = edge || window > 0;
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          float x = st[t][r] * sc;
          if constexpr (EXT == 2) x = tanhf(x) * (softcap * LOG2E);
          if (edge) {
            const int kv = kv0 + t * 32 + 8 * (r >> 2) + 4 * hf + (r & 3);
            bool ok = kv <= qpos && kv < len;
            if constexpr (EXT > 0) ok = ok && (window <= 0 || kv > qpos - window);
            x = ok ? x : -INFINITY;
          }
          st[t][r] = x;
          mx = fmaxf(mx, x);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE_SIZE));
      if (__any(mx > m + SLACK)) {
        const float nm = fmaxf(m, mx);
        const float corr =
            nm == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - nm);
        m = nm;
        l *= corr;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= corr;
      }
      const float base = m == -INFINITY ? 0.f : m;
      u32x4 pf[4];
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float a = __builtin_amdgcn_exp2f(
              st[t >> 1][(t & 1) * 8 + w * 2] - base);
          const float b = __builtin_amdgcn_exp2f(
              st[t >> 1][(t & 1) * 8 + w * 2 + 1] - base);
          sum += a + b;
          pf[t][w] = pack_bf16(a, b);
        }
      l += sum;
      // O^T += V^T P^T
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const unsigned short* at = vt + (n * 32 + lc) * VT_ROW;
          const u32x2 a = *reinterpret_cast<const u32x2*>(
              at + ((t * 4 + hf) ^ (2 * (n & 3))) * 4);
          const u32x2 b = *reinterpret_cast<const u32x2*>(
              at + ((t * 4 + 2 + hf) ^ (2 * (n & 3))) * 4);
          o[n] = mfma32x32x16_bf16(u32x4{a[0], a[1], b[0], b[1]}, pf[t], o[n]);
        }
    }
    if (more) stash(lds + ((kt - kt0 + 1) & 1) * BUF);
    __syncthreads();
  }

  // normalise; a SINK logit joins the denominator only
  l += __shfl_xor(l, 32, WAVE_SIZE);
  float num = 1.f;
  if constexpr (EXT > 0) {
    if (sinks != nullptr) {
      const float sk = sinks[qh] * LOG2E;
      const float M = fmaxf(m, sk);
      num = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
      l = l * num + __builtin_amdgcn_exp2f(sk - M);
    }
  }
  const float inv = l > 0.f ? num / l : 0.f;
  store_rows<DVK>(out, lds + wave * 32 * DVK, o, inv, row0, q0 + wave * 32, nnew,
                  Hq, qh, lane);
}

// The same attention without options for heads of 128 channels: whole prompts
// and rows behind a history.
//  - keys and values go from memory into the LDS by themselves
//    (global_load_lds, 16 bytes a lane), rows as they are: no staging registers,
//    no LDS writes and no packing. Chunks are permuted through the lanes'
//    addresses: 16-byte chunks of a key row XORed with the row, 64-byte chunks
//    of a value row with row & 3. V^T comes out of the LDS by the transposing
//    read (ds_read_b64_tr_b16: 16 lanes read 4 keys x 16 channels and get 4 keys
//    of a channel each), conflict-free with that order.
//  - the waits for the loads are in `advance`.
//  - a wave works on 32 keys at a time: the scores of the next 32 are
//    multiplied while the exponentials of these 32 run, and the maximum of the
//    next is taken beside the second product, so that the matrix cores need not
//    wait for the softmax. For that the K buffer of tile j holds keys
//    64 j + 32 .. 64 j + 95, and the first 32 keys are multiplied before the
//    loop. Whole unmasked tiles run two to a turn without a branch but the
//    rescaling one; the rest, masked, 32 keys to a turn.
//  - scores stay unscaled; the factor is in the exponential's fma.
// Bound by the LDS reads (32 KB a wave and tile, half of the LDS rate at
// 1000 TFLOP/s) and the products: 32 heads on 8, one prompt of 7999 rows 638 ->
// 480 us (822 -> 1091 TFLOP/s), 2039 rows behind 6001 301 -> 233 (1007), 32 x 256
// 60 -> 52, 77 rows 8.8 -> 7.1, 33 rows behind 1000 38 -> 23, one row 5.7 -> 4.5.
// Eight waves on 256 rows: 493 and 238. An order of the instructions given with
// sched_group_barrier: 486 to 547. Of the long prompt the matrix cores are 58 % busy, at
// the 1.75 GHz that the card's power leaves. One wave a SIMD on 64 rows, which reads half
// as much from the LDS: 521; alone it issues an instruction every 5.5 cycles.
typedef __attribute__((ext_vector_type(4))) short s16x4;

DEVICE_INLINE u32x2 lds_read_tr(const unsigned short* p) {
  return __builtin_bit_cast(
      u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                 (__attribute__((address_space(3))) s16x4*)p));
}

// The tile of this workgroup, two of which run on a CU. The tiles with the most keys
// start first; but where one launch fills the chip no more than twice over, workgroups i
// and 256 + i share a CU from the start to the end: the first 256 then begin with the
// smallest of them, next to the largest of the others. us, largest first / so: 32 heads,
// two prompts of 1024 rows 34.5 / 29.4, four of 512 22.8 / 20.5, one of 2039 48.1 / 47.2
// (behind 6001 245 / 238, 2048 behind 2000 113 / 108), 16 heads, 4000 rows 85.4 / 83.8,
// 8 heads, 7999 158 / 155. Heads that do not divide 256 gain or lose by the list (28
// heads, 2039 rows 45.4 / 43.9, three prompts of 700 24.6 / 26.0) and stay. Several
// prompts lie in the batch's order, not by size, and gain or lose by that: of 43 drawn
// batches 1.00 of the time, .79 (six of 231 rows behind 0 to 4000 113 / 89) to 1.16 (1354
// and five of 48 to 506 32 / 37); of 35 single prompts .98, .96 to 1.04.
DEVICE_INLINE int tile_of(int Hq) {
  const int n = gridDim.x / Hq, at = blockIdx.x / Hq, chip = 256 / Hq;
  const bool twice = 256 % Hq == 0 && n > chip && n <= 2 * chip;
  return twice && at < chip ? n - chip + at : n - 1 - at;
}

template <bool PAGED>
__global__ __launch_bounds__(PF_THREADS, 2) void flash_rows_kernel(
    unsigned short* __restrict__ out,      // [T, Hq, 128]
    const unsigned short* __restrict__ q, const unsigned short* __restrict__ k,
    const unsigned short* __restrict__ v,
    const int* __restrict__ block_tables,  // [nseq, maxb]
    const int* __restrict__ tile_start, const int* __restrict__ tile_q0,
    const int* __restrict__ tile_hist, const int* __restrict__ tile_new,
    const int* __restrict__ tile_seq, int Hq, int Hkv, int maxb, float scale,
    long qs, long ks, long vs) {
  constexpr int D = 128, QK = D / 16, NT = D / 32;
  constexpr int TILE = BK * D;             // elements of a buffer
  constexpr int RW = BK / PF_WAVES;        // rows of a tile a wave brings
  constexpr int NI = RW / 4;               // instructions, 4 rows each
  constexpr int HB = 32;                   // keys of a turn
  static_assert(RW == PP_BS, "a wave brings one page");
  __shared__ __attribute__((aligned(1024))) unsigned short lds[4 * TILE];

  int qh = blockIdx.x % Hq;
  if (Hq % 8 == 0) qh = (qh % 8) * (Hq / 8) + qh / 8;
  const int tile = tile_of(Hq);
  const int kvh = qh / (Hq / Hkv);
  const int row0 = tile_start[tile];
  const int q0 = tile_q0[tile];
  if (q0 % BQ != 0) return;          // the second half of a list of 64-row tiles
  const int hist = PAGED ? tile_hist[tile] : 0;
  const int nnew = tile_new[tile];
  const int len = hist + nnew;
  const int* bt = PAGED ? block_tables + (long)tile_seq[tile] * maxb : nullptr;

  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int lc = lane & 31, hf = lane >> 5;

  const int qrow = q0 + wave * 32 + lc;            // within the new rows
  const int qpos = hist + qrow;
  u32x4 qf[QK];
  {
    const unsigned short* qp =
        q + (long)(row0 + min(qrow, nnew - 1)) * qs + (long)qh * D + hf * 8;
#pragma unroll
    for (int kk = 0; kk < QK; ++kk)
      qf[kk] = *reinterpret_cast<const u32x4*>(qp + kk * 16);
  }

  float m = -INFINITY, l = 0.f;                    // m in powers of two
  f32x16 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  const int lo_wave = hist + q0 + wave * 32;       // this wave's first row
  const bool idle = q0 + wave * 32 >= nnew;        // it has none
  const int kv_end = min(len, hist + q0 + BQ);     // causal bound
  const int nt = (kv_end + BK - 1) / BK;
  const float sc = scale * LOG2E;

  // the lanes' byte offsets in a wave's RW rows
  const int lr = lane >> 4, ch = lane & 15;
  const int r0 = wave * RW;
  const int kstep = PAGED ? D : (int)ks, vstep = PAGED ? D : (int)vs;
  unsigned int koffs[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
    koffs[i] = (unsigned)((i * 4 + lr) * kstep +
                          (ch ^ ((r0 + i * 4 + lr) & 15)) * 8) * 2;
  const unsigned int voffs = (unsigned)(lr * vstep + (ch ^ (lr << 2)) * 8) * 2;
  // keys (or values) key0 .. key0 + 63 into a buffer; rows behind the
  // sequence's end repeat its last, rows in front of its start stay out
  auto stage = [&](bool isk, int key0, unsigned short* to) {
    const int kv0 = key0 + r0;
    if (kv0 < 0) return;
    const int at = min(kv0, len - 1);
    const int step = isk ? kstep : vstep;
    const unsigned short* base;
    if constexpr (PAGED)
      base = (isk ? k : v) +
             (((long)bt[at / PP_BS] * Hkv + kvh) * PP_BS + at % PP_BS) * D;
    else
      base = (isk ? k + (long)(row0 + at) * ks : v + (long)(row0 + at) * vs) +
             (long)kvh * D;
    to += r0 * D;
    if (kv0 + RW <= len) {
#pragma unroll
      for (int i = 0; i < NI; ++i)
        load_to_lds(isk ? base : base + i * 4 * step, isk ? koffs[i] : voffs,
                    to + i * 4 * D);
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int row = i * 4 + lr;
        const int c = isk ? ch ^ ((r0 + row) & 15) : ch ^ (lr << 2);
        load_to_lds(base, (unsigned)(min(row, len - 1 - at) * step + c * 8) * 2,
                    to + i * 4 * D);
      }
    }
  };
  auto kbuf = [&](int j) { return lds + (j & 1) * TILE; };
  auto vbuf = [&](int j) { return lds + (2 + (j & 1)) * TILE; };

  // LDS places of the operands: K chunk kk, V channels 32 n
  const int koff = lc * D + ((hf ^ (lc & 15)) * 8);
  const int vrow = (lane & 15) >> 2;               // and its row & 3
  const int voff =
      (4 * hf + vrow) * D + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  const unsigned short *ka[QK], *va[NT];
#pragma unroll
  for (int i = 0; i < QK; ++i) ka[i] = lds + (koff ^ (i * 16));
#pragma unroll
  for (int i = 0; i < NT; ++i) va[i] = lds + 2 * TILE + voff + ((i ^ vrow) * 32);

  auto scores = [&](int at, f32x16& s) {           // at: elements from ka
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int kk = 0; kk < QK; ++kk)
      s = mfma32x32x16_bf16(*reinterpret_cast<const u32x4*>(ka[kk] + at),
                            qf[kk], s);
  };
  auto row_max = [&](const f32x16& s) {            // in powers of two
    float x = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) x = fmaxf(fmaxf(x, s[r]), s[r + 1]);
    x = fmaxf(x, s[15]);
    return half_wave_max(x) * sc;
  };
  auto rescale = [&](float mx) {
    if (__any(mx > m + SLACK)) {
      const float nm = fmaxf(m, mx);
      const float corr =
          nm == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - nm);
      m = nm;
      l *= corr;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] *= corr;
    }
    return m == -INFINITY ? 0.f : m;
  };
  auto weights = [&](const f32x16& s, u32x4 (&pf)[2], float base) {
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float a = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[t * 8 + w * 2], sc, -base));
        const float b = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[t * 8 + w * 2 + 1], sc, -base));
        sum += a + b;
        pf[t][w] = pack_bf16(a, b);
      }
    l += sum;
  };
  auto weigh = [&](int at, const u32x4 (&pf)[2]) {  // at: elements from va
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const unsigned short* p = va[n] + at + t * 16 * D;
        const u32x2 a = lds_read_tr(p), b = lds_read_tr(p + 8 * D);
        o[n] = mfma32x32x16_bf16(u32x4{a[0], a[1], b[0], b[1]}, pf[t], o[n]);
      }
  };
  // Tile j is in the LDS for every wave, and every wave is done with tile
  // j - 1, whose buffers tile j + 1 takes.
  auto advance = [&](int j) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if ((j + 1) * BK + HB < kv_end) stage(true, (j + 1) * BK + HB, kbuf(j + 1));
    if (j + 1 < nt) stage(false, (j + 1) * BK, vbuf(j + 1));
  };

  stage(true, HB - BK, kbuf(1));
  if (HB < kv_end) stage(true, HB, kbuf(0));
  stage(false, 0, vbuf(0));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  f32x16 st;
  scores(TILE + HB * D, st);

  // whole tiles, which no row of the wave needs a mask for
  const int full = idle ? 0 : min(nt - 1, (lo_wave + 1) / BK);
  float mx = full > 1 ? row_max(st) : 0.f;
  auto whole = [&](int j, int p) {                 // p = j & 1, a constant
    advance(j);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float base = rescale(mx);
      f32x16 next;
      u32x4 pf[2];
      scores(p * TILE + h * HB * D, next);
      weights(st, pf, base);
      weigh(p * TILE + h * HB * D, pf);
      st = next;
      mx = row_max(st);
    }
  };
  int j = 0;
  for (; j + 1 < full; j += 2) {
    whole(j, 0);
    whole(j + 1, 1);
  }
  for (; j < nt; ++j) {
    advance(j);
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int kv0 = j * BK + h * HB;
      if (kv0 > lo_wave + 31 || kv0 >= kv_end || idle) break;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kv = kv0 + 8 * (r >> 2) + 4 * hf + (r & 3);
        st[r] = kv <= qpos && kv < len ? st[r] : -INFINITY;
      }
      const float base = rescale(row_max(st));
      const int at = (j & 1) * TILE + h * HB * D;
      u32x4 pf[2];
      weights(st, pf, base);
      if (kv0 + HB < kv_end) scores(at, st);
      weigh(at, pf);
    }
  }
  __syncthreads();

  l += __shfl_xor(l, 32, WAVE_SIZE);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  store_rows<D>(out, lds + wave * 32 * D, o, inv, row0, q0 + wave * 32, nnew, Hq,
                qh, lane);
}

template <int D, int DVK, int EXT, bool PAGED>
void launch(void* out, const void* q, const void* k, const void* v,
            const int* bt, const int* start, const int* q0, const int* hist,
            const int* nnew, const int* seq, int ntiles, int Hq, int Hkv,
            int maxb, float scale, long qs, long ks, long vs,
            const float* sinks, int window, float softcap, hipStream_t s) {
  if (ntiles == 0) return;
  // Rows that the loads to the LDS can take: aligned to them, offsets within 32
  // bits; and a factor that a maximum of unscaled scores may be taken under.
  // It was the faster one at every size measured (above).
  if constexpr (D == 128 && DVK == 128 && EXT == 0) {
    const unsigned long at = (unsigned long)k | (unsigned long)v |
                             (unsigned long)(ks * 2) | (unsigned long)(vs * 2);
    constexpr long FAR = 1l << 24;
    if (at % 16 == 0 && ks >= 0 && vs >= 0 && ks < FAR && vs < FAR &&
        scale > 0.f) {
      hipLaunchKernelGGL((flash_rows_kernel<PAGED>), dim3((unsigned)ntiles * Hq),
                         dim3(PF_THREADS), 0, s, (unsigned short*)out,
                         (const unsigned short*)q, (const unsigned short*)k,
                         (const unsigned short*)v, bt, start, q0, hist, nnew,
                         seq, Hq, Hkv, maxb, scale, qs, ks, vs);
      return;
    }
  }
  hipLaunchKernelGGL((flash_prefill_kernel<D, DVK, EXT, PAGED>),
                     dim3((unsigned)ntiles * Hq), dim3(PF_THREADS), 0, s,
                     (unsigned short*)out, (const unsigned short*)q,
                     (const unsigned short*)k, (const unsigned short*)v, bt,
                     start, q0, hist, nnew, seq, Hq, Hkv, maxb, scale, qs, ks,
                     vs, sinks, window, softcap);
}

}  // namespace

void flash_prefill_paged_launch(
    void* out, const void* q, const void* kc, const void* vc,
    const int* block_tables, const int* tile_qstart, const int* tile_q0,
    const int* tile_hist, const int* tile_new, const int* tile_seq,
    int ntiles, int Hq, int Hkv, int D, int maxb, float scale, long qs,
    const float* sinks, int window, float softcap, int* err_unsupported,
    hipStream_t s) {
  *err_unsupported = 0;
  if ((D != 128 && D != 64 && D != 256) || Hq % Hkv != 0) {
    *err_unsupported = 1;
    return;
  }
#define PPG_FORM(DD, E)                                                       \
  launch<DD, DD, E, true>(out, q, kc, vc, block_tables, tile_qstart, tile_q0, \
                          tile_hist, tile_new, tile_seq, ntiles, Hq, Hkv,     \
                          maxb, scale, qs, 0, 0, sinks, window, softcap, s)
#define PPG_LAUNCH(DD)                                                        \
  if (softcap > 0.f) PPG_FORM(DD, 2);                                         \
  else if (sinks != nullptr || window > 0) PPG_FORM(DD, 1);                   \
  else PPG_FORM(DD, 0);
  if (D == 128) { PPG_LAUNCH(128) }
  else if (D == 64) { PPG_LAUNCH(64) }
  else { PPG_LAUNCH(256) }
#undef PPG_LAUNCH
#undef PPG_FORM
}

void flash_prefill_launch(void* out, const void* q, const void* k,
                          const void* v, const int* tile_start,
                          const int* tile_q0, const int* tile_len, int ntiles,
                          int Hq, int Hkv, int D, int DV, float scale,
                          long qs, long ks, long vs, const float* sinks,
                          int window, float softcap, int* err_unsupported,
                          hipStream_t s) {
  *err_unsupported = 0;
  const bool mla_dims = (D == 192 && DV == 128);
  if (((D != 128 && D != 64 && D != 256) && !mla_dims)
      || (!mla_dims && DV != D) || Hq % Hkv != 0) {
    *err_unsupported = 1;
    return;
  }
#define PF_FORM(DD, E, DVV)                                                   \
  launch<DD, DVV, E, false>(out, q, k, v, nullptr, tile_start, tile_q0,       \
                            nullptr, tile_len, nullptr, ntiles, Hq, Hkv, 0,   \
                            scale, qs, ks, vs, sinks, window, softcap, s)
#define PF_LAUNCH(DD)                                                         \
  if (softcap > 0.f) PF_FORM(DD, 2, DD);                                      \
  else if (sinks != nullptr || window > 0) PF_FORM(DD, 1, DD);                \
  else PF_FORM(DD, 0, DD);
  if (mla_dims) {
    // MLA expand-prefill (DeepSeek): 192-dim qk over 128-dim values
    PF_FORM(192, 0, 128);
  } else if (D == 128) { PF_LAUNCH(128) }
  else if (D == 64) { PF_LAUNCH(64) }
  else { PF_LAUNCH(256) }
#undef PF_LAUNCH
#undef PF_FORM
}

// ---------------------------------------------------------------------------
// MFMA layout probe: D = A[16x32] * B[32x16] on the 16x16x32 form, with the
// fragment layouts that decode attention and the products of few rows assume
// (the 32x32x16 form above is checked by the attention itself). Random
// asymmetric inputs against torch.matmul show a transposed fragment.
// ---------------------------------------------------------------------------
namespace {
__global__ void mfma_probe_kernel(float* __restrict__ d,
                                  const unsigned short* __restrict__ a,
                                  const unsigned short* __restrict__ b) {
  const int lane = threadIdx.x & 63;
  const int lc = lane & 15, lg = lane >> 4;
  u16x8 af, bf;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    af[j] = a[lc * 32 + lg * 8 + j];   // A[row=lc][k=lg*8+j]
    bf[j] = b[(lg * 8 + j) * 16 + lc]; // B[k=lg*8+j][col=lc]
  }
  f32x4 c{0.f, 0.f, 0.f, 0.f};
  c = mfma16x16x32_bf16(af, bf, c);
#pragma unroll
  for (int r = 0; r < 4; ++r) d[(lg * 4 + r) * 16 + lc] = c[r];
}
}  // namespace

void mfma_probe_launch(float* d, const void* a, const void* b, hipStream_t s) {
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, s, d,
                     (const unsigned short*)a, (const unsigned short*)b);
}
