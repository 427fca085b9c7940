// Paged-attention decode for MI355X (gfx950) — the TPOT-dominant kernel.
//
// Single new token per sequence attends over the paged KV cache.
// Replaces what the reference delegates to vLLM's paged_attention kernels;
// designed for CDNA4 rather than ported:
//
//  - a workgroup owns (sequence, kv head, part of the keys); the GQ = Hq/Hkv
//    query heads of a kv head share its K/V stream, so each KV byte is read
//    exactly once per step. The keys of a sequence are cut into parts when
//    (sequences x kv heads) alone leaves CUs without work (decode_parts);
//    a second kernel joins the parts where more than one has keys.
//  - 4 waves per workgroup, each with keys of its own, 16 or 32 a step (pages of 16);
//    parts of up to 64 keys are one page a wave, one step. Scores are
//    a matrix product, S^T = K Q^T on mfma_f32_16x16x32_bf16: K rows are the
//    A operand as they lie in the page, the GQ query
//    rows (zero rows up to 16) the B operand. One lane then holds one head's
//    scores of 4 keys a page, so maximum and sum take two cross-lane steps per 32
//    keys instead of four per key.
//  - probabilities stay fp32. paged_attn_decode_kernel multiplies them with the values
//    on the matrix cores, in three parts; paged_attn_heads_kernel, for one query head a
//    kv head and some of two of 64 channels, with fp32 FMA.
//  - fp8 keys become bf16 exactly (e4m3 has 3 mantissa bits) in registers.
//
// Bound by the K/V stream where the chip is full (5.3 to 5.5 TB/s), else by the longest
// part's chain: 1.9 us a step of 128 keys where nothing else runs.
//
// KV pool layout: [num_blocks, Hkv, BS, D] bf16 | fp8, BS = 16 tokens.
#include "common.h"

#include <type_traits>

// parts of a sequence, a part's keys, and the query heads of a workgroup: one or two
// (paged_attn_heads_kernel), or 0, all of a kv head (paged_attn_decode_kernel)
struct DecodeParts { int n, least, heads; };

// The step's rows as they leave the projection, where the kernel norms, rotates and
// stores them itself: q | k | v in bf16, or (rows null) as fp32 parts of it.
struct NewRows {
  const unsigned short* rows;         // [N, (Hq + 2 Hkv) * D]
  const float* parts;                 // [nparts, N, (Hq + 2 Hkv) * D]
  int nparts;
  const unsigned short *q_norm, *k_norm;   // [D] or null
  const float* cos_sin;               // [positions, D]
  const long *positions, *slots;      // [N]
  float eps;
};

namespace {

constexpr int BS = 16;       // tokens per KV block (page)
constexpr int NWAVES = 4;    // waves per workgroup
constexpr int THREADS = NWAVES * WAVE_SIZE;
constexpr int STEP = 32;     // keys per wave and step (two pages)
constexpr float LOG2E = 1.4426950408889634f;

typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(2))) int i32x2;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

// `n` bytes as 32-bit words, loaded in the widest pieces
template <int WORDS>
DEVICE_INLINE void load_words(unsigned int* dst, const void* src) {
  if constexpr (WORDS >= 4) {
#pragma unroll
    for (int i = 0; i < WORDS / 4; ++i) {
      const u32x4 v = reinterpret_cast<const u32x4*>(src)[i];
#pragma unroll
      for (int j = 0; j < 4; ++j) dst[i * 4 + j] = v[j];
    }
  } else if constexpr (WORDS == 2) {
    const u32x2 v = *reinterpret_cast<const u32x2*>(src);
    dst[0] = v[0];
    dst[1] = v[1];
  } else {
    dst[0] = *reinterpret_cast<const unsigned int*>(src);
  }
}

// four fp8 -> four f32
DEVICE_INLINE void fp8x4_f32(unsigned int w, float* o) {
  const f32x2 a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false);
  const f32x2 b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w, true);
  o[0] = a[0]; o[1] = a[1]; o[2] = b[0]; o[3] = b[1];
}

// the high halves of two f32 as one word of bf16 (exact when the low halves
// are zero)
DEVICE_INLINE unsigned int pack_hi(float lo, float hi) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(unsigned int, hi),
                               __builtin_bit_cast(unsigned int, lo),
                               0x07060302u);
}
DEVICE_INLINE float high_half(float v) {
  return __builtin_bit_cast(float,
                            __builtin_bit_cast(unsigned int, v) & 0xffff0000u);
}

// The fp32 number below one that is positive; 0 of 0, a NaN of a NaN. The high half of
// it, taken from the number, leaves more than nothing and no more than 17 bits, and
// once more of that no more than 8: three parts, none of which is 0 (down to 2^-94),
// so that an infinite value times them is that infinity and no NaN.
DEVICE_INLINE float next_below(float v) {
  return __builtin_bit_cast(
      float, __builtin_elementwise_sub_sat(__builtin_bit_cast(unsigned int, v), 1u));
}

// eight fp8 -> eight bf16 (exact)
DEVICE_INLINE u32x4 fp8x8_bf16(u32x2 w) {
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    o[i * 2] = __builtin_bit_cast(
        unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, false));
    o[i * 2 + 1] = __builtin_bit_cast(
        unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w[i], 1.f, true));
  }
  return o;
}

DEVICE_INLINE f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(s16x8, a),
                                                 __builtin_bit_cast(s16x8, b), c,
                                                 0, 0, 0);
}

// Sums and maxima over the key groups without the LDS: as shuffles these exchanges, most
// of them in the sums at the end, were 12 % of the kernel over 240 shapes (16 heads of
// 256, us: 512 x 40 keys 53.6 -> 42.0, one x 300 12.2 -> 11.1; 32 of 128: 64 x 400 21.0
// -> 19.2).
DEVICE_INLINE float sum_groups(float v) {
  f32x2 p = with_lane<16>(v);
  p = with_lane<32>(p[0] + p[1]);
  return p[0] + p[1];
}
DEVICE_INLINE float max_groups(float v) {
  f32x2 p = with_lane<16>(v);
  p = with_lane<32>(fmaxf(p[0], p[1]));
  return fmaxf(p[0], p[1]);
}

// keys per part of a sequence of `len` tokens: whole steps, at least `least`
DEVICE_INLINE int part_tokens(int len, int nsplit, int least) {
  const int per = (len + nsplit - 1) / nsplit;
  return max((per + STEP - 1) / STEP * STEP, least);
}

DEVICE_INLINE int window_start(int len, int window) {
  return window > 0 && len > window ? len - window : 0;
}

// One query head a kv head (and pools that the other kernel's direct loads do not take):
// its weighted sums are one fp32 FMA a value, fewer
// instructions than the products below, of whose 16 rows 15 would be empty, and
// nothing goes through the LDS but the weights. Against those, us: 403 x 35 keys, 32
// heads of 128 63 / 69, 72 x 39 14.9 / 16.6, 31 x 37 in fp8 6.6 / 8.3; 64 channels
// in fp8, 476 x 1150 in a window of 128 63 / 79. (Of 36 batches of 128 channels the
// products would be the faster ones by 5 % on average, 9 of them slower, to 1.27.)
// Two heads of 64 channels (GQ = 2), us, this / those: 16 on 8 in fp8, 8 x 20 to 64 keys
// behind a wide table 4.8 / 5.7, 384 11.0 / 14.8, 8 x 200 to 400 6.0 / 7.1, 128 x 500 to
// 1200 30.9 / 28.1; 8 x 20 to 64 behind a table of 64 3.4 / 4.0, in bf16 too.
//  - probabilities go through LDS to a layout of 16 lanes a value row (D/16 channels
//    each) x 4 keys, where the weighted sum is fp32 FMA on values loaded 16 bytes
//    (bf16) or 8 bytes (fp8) a lane.
template <int D, int GQ, bool FP8, bool EXT>
__global__ __launch_bounds__(THREADS, D == 64 ? 5 : D == 256 ? (FP8 ? 3 : 2) : 4)
void paged_attn_heads_kernel(
    unsigned short* __restrict__ out,        // [N, Hq, D]
    const unsigned short* __restrict__ q,    // [N, Hq, D]
    const char* __restrict__ kc,             // [B, Hkv, BS, D] bf16|fp8
    const char* __restrict__ vc,             // [B, Hkv, BS, D]
    const int* __restrict__ block_tables,    // [N, max_blocks]
    const int* __restrict__ seq_lens,        // [N]
    float* __restrict__ part,                // [N, Hq / GQ, nsplit, GQ, D + 2]
    int least,                               // keys of a part (part_tokens)
    int Hkv, int rep, int max_blocks, float scale, long q_stride,
    const float* __restrict__ sinks,         // [Hq] or null (GPT-OSS)
    int window,                              // 0 = full attention
    float softcap) {                         // 0 = off (Gemma-2 tanh cap)
  constexpr int DV = D / 16;        // value channels per lane
  constexpr int ES = FP8 ? 1 : 2;   // bytes per cached number
  constexpr int QK = D / 32;        // products per 16 keys
  constexpr int KW = 8 * ES / 4;    // words of a K fragment
  constexpr int VW = DV * ES / 4;   // words of a lane's value channels
  static_assert(D == 64 || D == 128 || D == 256, "D in {64, 128, 256}");

  const int seq = blockIdx.x;
  const int h = blockIdx.y;         // GQ query heads; rep of these share a kv head
  const int hk = rep == 1 ? h : h / rep;
  const int nsplit = gridDim.z;
  const int Hq = gridDim.y * GQ;
  const int len = seq_lens[seq];
  // sliding window (EXT): the query sits at position len - 1 and attends
  // [max(0, len - window), len); the parts cut only that
  const int wstart = EXT ? window_start(len, window) : 0;
  const int from = wstart / BS * BS;
  const int span = part_tokens(len - from, nsplit, least);
  const int t0 = from + (int)blockIdx.z * span;
  const int t1 = min(len, t0 + span);
  if (nsplit > 1 && t0 >= len) return;     // the join skips it as well
  // the only part with keys is the result (one x 60 keys 8.5 -> 7.8)
  const bool whole = nsplit == 1 || span >= len - from;

  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int wave = threadIdx.x / WAVE_SIZE;
  const int g = lane >> 4;          // key group / k-slot group
  const int sub = lane & 15;        // head (scores), channel slice (values)

  __shared__ float lds_p[NWAVES][STEP][GQ];
  __shared__ float lds_c[NWAVES][GQ];
  __shared__ float lds_acc[NWAVES][GQ][D];
  __shared__ float lds_ms[NWAVES][GQ][2];

  // Q as the B operand: column `sub` = head, rows g*8 .. g*8+7 of each chunk
  u16x8 qf[QK];
#pragma unroll
  for (int kk = 0; kk < QK; ++kk) {
    u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
    if (sub < GQ)
      z = *reinterpret_cast<const u16x8*>(
          q + (long)seq * q_stride + ((long)h * GQ + sub) * D + kk * 32 + g * 8);
    qf[kk] = z;
  }

  float m = -INFINITY, s = 0.f;     // of head `sub`; s: this lane's keys
  float acc[GQ][DV];
#pragma unroll
  for (int gq = 0; gq < GQ; ++gq)
#pragma unroll
    for (int j = 0; j < DV; ++j) acc[gq][j] = 0.f;

  const char* kbase = kc + (long)hk * BS * D * ES;
  const char* vbase = vc + (long)hk * BS * D * ES;
  const long page_bytes = (long)Hkv * BS * D * ES;
  const int* bt = block_tables + (long)seq * max_blocks;
  const int last_page = (len - 1) / BS;
  const float sc = scale * LOG2E;

  auto step = [&](auto pages, int c0) {
    constexpr int PG = decltype(pages)::value, VR = 4 * PG;
    const int page = c0 / BS;
    long at[PG];
#pragma unroll
    for (int p = 0; p < PG; ++p)
      at[p] = (long)bt[min(page + p, last_page)] * page_bytes;
    unsigned int kw[PG][QK][KW], vw[VR][VW];
#pragma unroll
    for (int p = 0; p < PG; ++p)
#pragma unroll
      for (int kk = 0; kk < QK; ++kk)
        load_words<KW>(kw[p][kk],
                       kbase + at[p] + (sub * D + kk * 32 + g * 8) * ES);
#pragma unroll
    for (int i = 0; i < VR; ++i)
      load_words<VW>(vw[i], vbase + at[i / 4] +
                                (((i & 3) * 4 + g) * D + sub * DV) * ES);

    // scores: lane = head `sub`, keys c0 + p*16 + g*4 + r
    float x[VR];
    float mx = -INFINITY;
#pragma unroll
    for (int p = 0; p < PG; ++p) {
      f32x4 st{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < QK; ++kk) {
        u32x4 a;
        if constexpr (FP8) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            float f[4];
            fp8x4_f32(kw[p][kk][w], f);
            a[w * 2] = pack_hi(f[0], f[1]);
            a[w * 2 + 1] = pack_hi(f[2], f[3]);
          }
        } else {
          a = u32x4{kw[p][kk][0], kw[p][kk][1], kw[p][kk][2], kw[p][kk][3]};
        }
        st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(s16x8, a), __builtin_bit_cast(s16x8, qf[kk]),
            st, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = c0 + p * 16 + g * 4 + r;
        float v = st[r] * sc;
        bool ok = tok < t1;
        if constexpr (EXT) {
          if (softcap > 0.f)
            v = tanhf(st[r] * scale / softcap) * (softcap * LOG2E);
          ok = ok && tok >= wstart;
        }
        v = ok ? v : -INFINITY;
        x[p * 4 + r] = v;
        mx = fmaxf(mx, v);
      }
    }
    mx = max_groups(mx);
    const float nm = fmaxf(m, mx);
    const float base = nm == -INFINITY ? 0.f : nm;
    const float corr = __builtin_amdgcn_exp2f(m - base);
    m = nm;
    s *= corr;
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      x[i] = __builtin_amdgcn_exp2f(x[i] - base);
      s += x[i];
    }
    if (sub < GQ) {
#pragma unroll
      for (int p = 0; p < PG; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          lds_p[wave][p * 16 + g * 4 + r][sub] = x[p * 4 + r];
      if (g == 0) lds_c[wave][sub] = corr;
    }
    // one wave's LDS operations stay in order; the compiler must keep them so
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (__any(sub < GQ && corr != 1.f)) {
#pragma unroll
      for (int gq = 0; gq < GQ; ++gq) {
        const float c = lds_c[wave][gq];
#pragma unroll
        for (int j = 0; j < DV; ++j) acc[gq][j] *= c;
      }
    }
    // values: lane = channels sub*DV .., keys (i/4)*16 + (i%4)*4 + g. Rows that
    // are not the sequence's (behind its end in its last page, in front of its
    // window) may hold anything, and a weight of 0 does not undo a NaN
    if (c0 + PG * BS > t1 || (EXT && c0 < wstart)) {
#pragma unroll
      for (int i = 0; i < VR; ++i) {
        const int tok = c0 + (i / 4) * 16 + (i & 3) * 4 + g;
        if (tok >= t1 || (EXT && tok < wstart))
#pragma unroll
          for (int w = 0; w < VW; ++w) vw[i][w] = 0;
      }
    }
#pragma unroll
    for (int i = 0; i < VR; ++i) {
      float pr[GQ], vf[DV];
#pragma unroll
      for (int gq = 0; gq < GQ; ++gq)
        pr[gq] = lds_p[wave][i * 4 + g][gq];
#pragma unroll
      for (int w = 0; w < VW; ++w) {
        if constexpr (FP8) {
          fp8x4_f32(vw[i][w], vf + w * 4);
        } else {
          vf[w * 2] = __builtin_bit_cast(float, vw[i][w] << 16);
          vf[w * 2 + 1] = __builtin_bit_cast(float, vw[i][w] & 0xffff0000u);
        }
      }
#pragma unroll
      for (int gq = 0; gq < GQ; ++gq)
#pragma unroll
        for (int j = 0; j < DV; ++j) acc[gq][j] += pr[gq] * vf[j];
    }
    asm volatile("" ::: "memory");  // P is read before the next step's writes
  };
  // a page for each wave where that is all (one step of latency, and no wave
  // without keys beside one with two pages), else two a step and a last one
  const bool few = t1 - t0 <= NWAVES * BS;
  int c0 = t0 + wave * (few ? BS : STEP);
  if (!few)
    for (; c0 + BS < t1; c0 += NWAVES * STEP)
      step(std::integral_constant<int, 2>{}, c0);
  if (c0 < t1) step(std::integral_constant<int, 1>{}, c0);

  // the four key groups of a wave, then the waves
  s = sum_groups(s);
#pragma unroll
  for (int gq = 0; gq < GQ; ++gq) {
#pragma unroll
    for (int j = 0; j < DV; ++j) {
      const float a = sum_groups(acc[gq][j]);
      if (g == 0) lds_acc[wave][gq][sub * DV + j] = a;
    }
  }
  if (g == 0 && sub < GQ) {
    lds_ms[wave][sub][0] = m;
    lds_ms[wave][sub][1] = s;
  }
  __syncthreads();

  for (int u = threadIdx.x; u < GQ * D; u += THREADS) {
    const int gq = u / D;
    const int d = u % D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) M = fmaxf(M, lds_ms[w][gq][0]);
    float extra = 0.f;
    if constexpr (EXT) {
      // an attention sink joins the softmax denominator only; with several
      // parts the join adds it
      if (sinks != nullptr && whole) {
        const float sk = sinks[h * GQ + gq] * LOG2E;
        M = fmaxf(M, sk);
        extra = __builtin_amdgcn_exp2f(sk - M);
      }
    }
    const float base = M == -INFINITY ? 0.f : M;
    float num = 0.f, den = extra;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
      const float wt = __builtin_amdgcn_exp2f(lds_ms[w][gq][0] - base);
      num += wt * lds_acc[w][gq][d];
      den += wt * lds_ms[w][gq][1];
    }
    if (whole) {
      out[((long)seq * Hq + (long)h * GQ + gq) * D + d] =
          f2bf(den > 0.f ? num / den : 0.f);
    } else {
      float* pp = part + ((((long)seq * gridDim.y + h) * nsplit + blockIdx.z) * GQ +
                          gq) * (D + 2);
      pp[d] = num;
      if (d == 0) {
        pp[D] = M;
        pp[D + 1] = den;
      }
    }
  }
}

// LDS of a wave: a step's pages of K and V
constexpr int ring_bytes(int D, bool fp8, int pages) {
  return 2 * pages * BS * D * (fp8 ? 1 : 2);
}

// Two to eight query heads a kv head. A wave streams keys of its own, PGS pages (16
// keys each) a step, K and V by direct loads into its ring in the LDS: the next
// step's K while these weights and values are multiplied, the next V while the next
// scores are, so that something is under way all the time, and no register holds a
// load (with K and V loaded to registers the compiler kept half of V back until K had
// come: a step cost two latencies, and prefetched by hand they spilled).
//  - scores S^T = K Q^T as above; a lane ends with the scores of one head and the
//    keys 4 g .. 4 g + 3 of each page, which is the operand of O^T = V^T P^T as it
//    lies: V^T comes out of the LDS by the transposing read in that order of keys.
//  - weights stay fp32: they are the sum of three bf16 parts (8 + 8 + 8 bits), each
//    multiplied with the values, which are bf16 numbers, exactly; sums in fp32. Three
//    products of 16 rows for 4 heads' 256 FMAs a lane and 32 keys.
//  - PGS: two pages a step where workgroups are few, one where many share a CU
//    (decode_pages).
// Bound by memory where the chip is full: 32 sequences of 3900 keys (32 heads on 8)
// 92 us, 5.5 TB/s, 512 x 1000 to 3000 758 (782 before, with fp32 FMA on loads to
// registers); of unequal lengths by the longest: 48 x 3500 to 7900 in fp8 135 -> 119,
// 64 x 200 to 2000 of 32 heads on 4 44 -> 33, 16 x 300 to 1200 20.4 -> 16.3, 4 x 2000
// to 6000 27 -> 20.7; 512 x 256 to 383 128 -> 125. Of 196 batches of 12 to 512
// sequences of 40 to 6000 keys none is slower by more than 3 %, .80 of the time on
// average; of 1536 of 1 to 384 sequences of 20 to 1200 keys 94 are, .82 on average, most
// of two heads a kv head and up to 64 keys (16 heads on 8 of 128, three x 20 to 64 3.9 ->
// 4.2, 128 in fp8 6.8 -> 7.5): a workgroup of one step is its latencies, of which the LDS
// adds one.
// EXT: sinks / sliding window / softcap (GPT-OSS and Gemma variants).
// NEW: q is not there yet, nor the step's own key and value in the pools. Each workgroup
// makes its query heads from the projection's row, and the one whose part ends with the
// sequence the kv head's key and value; it stores them and, since its loads from the pool
// are under way, puts them over the row that these bring into the LDS. All of it, in the
// order and to the bit of the row kernel (qkv_store), while the first pages come, so that
// a launch and a round trip are saved. us, in two launches / in one, 32 heads on 8: one
// row of 1000 keys 9.5 / 8.0, 16 of 300 to 1200 19.1 / 16.5, 512 of 256 to 383 139.9 /
// 131.9, 48 of 3500 to 7900 in fp8 125.4 / 124.2; 64 x 200 to 2000 of 32 on 4 with norms
// 38.0 / 36.2. Where a CU works through many workgroups of one step each, the row's
// chain stands in front of every one: 512 x 40 to 58 36.8 / 40.7, in fp8 34 / 42.
template <int D, bool FP8, bool EXT, int PGS, bool NEW>
__global__ __launch_bounds__(THREADS, D == 256 || ring_bytes(D, FP8, PGS) > 8192 ? 2
                                    : D == 64 && PGS == 1                      ? 5 : 3)
void paged_attn_decode_kernel(
    unsigned short* __restrict__ out,        // [N, Hq, D]
    const unsigned short* __restrict__ q,    // [N, Hq, D]
    const char* __restrict__ kc,             // [B, Hkv, BS, D] bf16|fp8
    const char* __restrict__ vc,             // [B, Hkv, BS, D]
    const int* __restrict__ block_tables,    // [N, max_blocks]
    const int* __restrict__ seq_lens,        // [N]
    float* __restrict__ part,                // [N, Hkv, nsplit, GQ, D + 2]
    int least,                               // keys of a part (part_tokens)
    int Hkv, int GQ, int max_blocks, float scale, long q_stride,
    const float* __restrict__ sinks,         // [Hq] or null (GPT-OSS)
    int window,                              // 0 = full attention
    float softcap,                           // 0 = off (Gemma-2 tanh cap)
    NewRows nr) {
  constexpr int RB = FP8 ? D : 2 * D;   // bytes of a row
  constexpr int CPR = RB / 16;          // 16-byte chunks of a row
  constexpr int RPI = 64 / CPR;         // rows of a load
  constexpr int PI = BS / RPI;          // loads of a page
  constexpr int PAGE = BS * RB;
  constexpr int QK = D / 32;            // products per 16 keys
  constexpr int VT = D / 16;            // tiles of 16 channels
  constexpr int OS = D + 4;             // fp32 row of the sums
  constexpr int NK = 4 * PGS;           // keys of a lane and step
  constexpr int RING = ring_bytes(D, FP8, PGS);
  static_assert(D == 64 || D == 128 || D == 256, "D in {64, 128, 256}");
  static_assert(RING >= 8 * OS * 4, "8 heads' sums");
  __shared__ __attribute__((aligned(1024))) char lds[NWAVES * RING];
  __shared__ float lds_ms[NWAVES][16][2];
  constexpr int QS = D + 8;             // row of q in the LDS
  __shared__ __attribute__((aligned(16))) unsigned short new_q[NEW ? 8 * QS : 8];
  __shared__ __attribute__((aligned(16))) char new_kv[2][NEW ? RB : 16];

  const int seq = blockIdx.x;
  const int h = blockIdx.y;         // kv head
  const int nsplit = gridDim.z;
  const int Hq = Hkv * GQ;
  const int lane = threadIdx.x & (WAVE_SIZE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE_SIZE);
  const int g = lane >> 4;          // key group / k-slot group
  const int sub = lane & 15;        // head; key (scores), channel (values) of a tile

  // Q as the B operand: column `sub` = head, rows g*8 .. g*8+7 of each chunk
  u32x4 qf[QK];
  if constexpr (!NEW) {
#pragma unroll
    for (int kk = 0; kk < QK; ++kk) {
      qf[kk] = *reinterpret_cast<const u32x4*>(
          q + (long)seq * q_stride + ((long)h * GQ + min(sub, GQ - 1)) * D +
          kk * 32 + g * 8);
    }
  }
  long pos = 0, slot = -1;
  if constexpr (NEW) {
    pos = nr.positions[seq];
    slot = nr.slots[seq];
  }

  // Orders of a row's chunks in the LDS, through the lanes' addresses, so that 16
  // keys of a chunk, and 8 (fp8: 16) keys of 16 channels, lie in different banks.
  auto key_chunk = [](int c, int row) {
    return c ^ (RB >= 256 ? row & 15 : RB == 128 ? (row >> 1) & 7 : (row >> 2) & 3);
  };
  auto value_chunk = [](int c, int row) {
    if (FP8)
      return RB == 256   ? c ^ (row & 15)
             : RB == 128 ? c ^ ((row >> 1) & 7) ^ (row >> 4 << 2)
                         : c ^ ((row >> 2) & 3);
    return c ^ (RB >= 256 ? (row & 7) << 1 : ((row >> 1) & 3) << 1);
  };
  unsigned int koff[PI], voff[2][PI];
#pragma unroll
  for (int i = 0; i < PI; ++i) {
    const int row = i * RPI + lane / CPR, c = lane % CPR;
    koff[i] = row * RB + key_chunk(c, row) * 16;
    voff[0][i] = row * RB + value_chunk(c, row) * 16;
    voff[1][i] = row * RB + value_chunk(c, row + BS) * 16;
  }
  // The pages of a first part that begins at key 0 come beside the length, the
  // lanes' offsets are made while both are on their way.
  const int* bt = block_tables + (long)seq * max_blocks;
  const int most = max_blocks - 1;
  int len = seq_lens[seq];
  int first[1 + PGS];
  first[0] = bt[min(wave, most)];
#pragma unroll
  for (int p = 0; p < PGS; ++p) first[1 + p] = bt[min(wave * PGS + p, most)];
#pragma unroll
  for (int i = 0; i < PI; ++i)
    asm volatile("" : "+v"(koff[i]), "+v"(voff[0][i]), "+v"(voff[1][i]));
  asm volatile("" : "+s"(len), "+s"(first[0]), "+s"(first[1]), "+s"(first[PGS])
               : "s"(kc), "s"(vc));
  // sliding window (EXT): the query sits at position len - 1 and attends
  // [max(0, len - window), len); the parts cut only that
  const int wstart = EXT ? window_start(len, window) : 0;
  const int from = wstart / BS * BS;
  const int span =
      nsplit > 1 ? part_tokens(len - from, nsplit, least) : len - from;
  const int t0 = from + (int)blockIdx.z * span;
  const int t1 = min(len, t0 + span);
  // the only part with keys is the result (one x 60 keys 8.5 -> 7.8)
  const bool whole = nsplit == 1 || span >= len - from;

  float m = -INFINITY, s = 0.f;     // of head `sub`; s: this lane's keys
  f32x4 acc[VT];                    // channels 16 i + 4 g .. of head `sub`
#pragma unroll
  for (int i = 0; i < VT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const char* kbase = kc + (long)h * PAGE;
  const char* vbase = vc + (long)h * PAGE;
  const long page_bytes = (long)Hkv * PAGE;
  const int last_page = (len - 1) / BS;
  const float sc = scale * LOG2E;

  char* kl = lds + wave * RING;
  char* vl = kl + PGS * PAGE;
  auto stage = [&](const char* base, const unsigned int* off, char* to) {
#pragma unroll
    for (int i = 0; i < PI; ++i)
      load_to_lds((const unsigned short*)base, off[i],
                  (const unsigned short*)(to + i * 1024));
  };
  auto stage_k = [&](const int* page, int np) {
    stage(kbase + page[0] * page_bytes, koff, kl);
    if (PGS > 1 && np > 1) stage(kbase + page[1] * page_bytes, koff, kl + PAGE);
  };
  auto stage_v = [&](const int* page, int np) {
    stage(vbase + page[0] * page_bytes, voff[0], vl);
    if (PGS > 1 && np > 1) stage(vbase + page[1] * page_bytes, voff[1], vl + PAGE);
  };
  auto wait = [&](int pages) {           // all but the youngest `pages` are there
    if (PGS > 1 && pages > 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PI) : "memory");
    else if (pages > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PI) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

  // a page for each wave where that is all (one step of latency, and no wave
  // without keys beside one with two pages), else two a step
  const int ps = t1 - t0 <= NWAVES * BS ? 1 : PGS;
  const int stride = NWAVES * ps * BS;
  int c0 = t0 + wave * ps * BS;
  auto pages_at = [&](int c) { return min(ps, (t1 - c + BS - 1) / BS); };
  int np = pages_at(c0);
  int page[2] = {0, 0}, next[2] = {0, 0};
  if (t0 == 0) {
    page[0] = ps == 1 ? first[0] : first[1];
    page[1] = first[PGS];
  } else {
#pragma unroll
    for (int p = 0; p < PGS; ++p) page[p] = bt[max(min(c0 / BS + p, last_page), 0)];
  }
  // the part that ends with the sequence stores its key and value
  const bool owner = len > 0 ? t0 < len && len <= t0 + span : blockIdx.z == 0;
  if (NEW && nsplit > 1 && t0 >= len && !owner) return;
  int last_block = 0;
  if constexpr (NEW) last_block = bt[max(last_page, 0)];
  // both are there before the loads that the compiler does not count
  asm volatile("" ::"s"(page[0]), "s"(page[1]));
  if constexpr (!NEW) {
#pragma unroll
    for (int kk = 0; kk < QK; ++kk) {
      asm volatile("" : "+v"(qf[kk]));
      if (sub >= GQ) qf[kk] = u32x4{0, 0, 0, 0};
    }
  }
  if (c0 < t1) {
    stage_k(page, np);
    stage_v(page, np);
  }
  if constexpr (NEW) {
    constexpr int LPH = D / 16, HALF = D / 2;   // lanes of a head: 8 channels twice
    const int u = threadIdx.x / LPH, c = threadIdx.x % LPH * 8;
    if (u < GQ + 2) {
      const int head = u < GQ ? h * GQ + u : Hq + (u - GQ) * Hkv + h;
      const long row = (long)(Hq + 2 * Hkv) * D, at = seq * row + head * D + c;
      const float* cs = nr.cos_sin + pos * D + c;
      u16x8 a, b;
      float co[8], si[8];
      if (u <= GQ) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          co[i] = cs[i];
          si[i] = cs[HALF + i];
        }
      }
      if (nr.rows != nullptr) {
        a = *reinterpret_cast<const u16x8*>(nr.rows + at);
        b = *reinterpret_cast<const u16x8*>(nr.rows + at + HALF);
      } else {
        a = join_parts8(nr.parts + at, gridDim.x * row, nr.nparts);
        b = join_parts8(nr.parts + at + HALF, gridDim.x * row, nr.nparts);
      }
      if (u <= GQ) {
        float x[8], y[8], o[8];
        bf8_to_f32(a, x);
        bf8_to_f32(b, y);
        const unsigned short* w = u < GQ ? nr.q_norm : nr.k_norm;
        if (w != nullptr) {
          float ss = 0.f, wx[8], wy[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) ss += x[i] * x[i] + y[i] * y[i];
#pragma unroll
          for (int i = LPH / 2; i >= 1; i >>= 1) ss += __shfl_xor(ss, i, 64);
          const float inv = rsqrtf(ss / D + nr.eps);
          bf8_to_f32(*reinterpret_cast<const u16x8*>(w + c), wx);
          bf8_to_f32(*reinterpret_cast<const u16x8*>(w + c + HALF), wy);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            x[i] *= inv * wx[i];
            y[i] *= inv * wy[i];
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          o[i] = x[i] * co[i] - y[i] * si[i];
          y[i] = y[i] * co[i] + x[i] * si[i];
        }
        a = f32_to_bf8(o);
        b = f32_to_bf8(y);
      }
      if (u < GQ) {
        *reinterpret_cast<u16x8*>(new_q + u * QS + c) = a;
        *reinterpret_cast<u16x8*>(new_q + u * QS + c + HALF) = b;
      } else {
        char* own = new_kv[u - GQ];
        char* pool = const_cast<char*>(u == GQ ? kc : vc);
        const bool store = owner && slot >= 0;
        const long to = ((slot / BS * Hkv + h) * BS + slot % BS) * D + c;
        if constexpr (FP8) {
          u8x8 qa, qb;
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            qa[i] = f32_to_fp8(bf2f(a[i]));
            qb[i] = f32_to_fp8(bf2f(b[i]));
          }
          *reinterpret_cast<u8x8*>(own + c) = qa;
          *reinterpret_cast<u8x8*>(own + c + HALF) = qb;
          if (store) {
            *reinterpret_cast<u8x8*>(pool + to) = qa;
            *reinterpret_cast<u8x8*>(pool + to + HALF) = qb;
          }
        } else {
          *reinterpret_cast<u16x8*>(own + c * 2) = a;
          *reinterpret_cast<u16x8*>(own + (c + HALF) * 2) = b;
          if (store) {
            *reinterpret_cast<u16x8*>(pool + to * 2) = a;
            *reinterpret_cast<u16x8*>(pool + (to + HALF) * 2) = b;
          }
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < QK; ++kk) {
      qf[kk] = *reinterpret_cast<const u32x4*>(new_q + min(sub, GQ - 1) * QS +
                                               kk * 32 + g * 8);
      if (sub >= GQ) qf[kk] = u32x4{0, 0, 0, 0};
    }
  }
  // whether the row stored is the sequence's last (a slot elsewhere, or none, leaves what
  // the pool holds there)
  const int last = len - 1;
  const bool mine = NEW && slot == (long)last_block * BS + last % BS;
  while (c0 < t1) {
    const int cn = c0 + stride;
    const int nn = cn < t1 ? pages_at(cn) : 0;
#pragma unroll
    for (int p = 0; p < PGS; ++p) next[p] = bt[min(cn / BS + p, last_page)];
    wait(np);
    const bool own = mine && c0 <= last && last < c0 + np * BS;
    if constexpr (NEW) {
      const int p = (last - c0) / BS, r = last % BS;
      if (own && lane < CPR)
        *reinterpret_cast<u32x4*>(kl + p * PAGE + r * RB + key_chunk(lane, r) * 16) =
            *reinterpret_cast<const u32x4*>(new_kv[0] + lane * 16);
    }
    // scores: lane = head `sub`, keys c0 + p*16 + g*4 + r
    f32x4 st[PGS];
#pragma unroll
    for (int p = 0; p < PGS; ++p) {
      st[p] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (p < np) {
#pragma unroll
        for (int kk = 0; kk < QK; ++kk) {
          u32x4 a;
          if constexpr (FP8)
            a = fp8x8_bf16(*reinterpret_cast<const u32x2*>(
                kl + p * PAGE + sub * RB +
                key_chunk(kk * 2 + (g >> 1), sub) * 16 + (g & 1) * 8));
          else
            a = *reinterpret_cast<const u32x4*>(
                kl + p * PAGE + sub * RB + key_chunk(kk * 4 + g, sub) * 16);
          st[p] = mfma16(a, qf[kk], st[p]);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the keys are read
    if (nn > 0) stage_k(next, nn);
    float x[NK], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int tok = c0 + (i >> 2) * 16 + g * 4 + (i & 3);
      float v = st[i >> 2][i & 3] * sc;
      bool ok = (i >> 2) < np && tok < t1;
      if constexpr (EXT) {
        if (softcap > 0.f)
          v = tanhf(st[i >> 2][i & 3] * scale / softcap) * (softcap * LOG2E);
        ok = ok && tok >= wstart;
      }
      x[i] = ok ? v : -INFINITY;
      mx = fmaxf(mx, x[i]);
    }
    mx = max_groups(mx);
    const float nm = fmaxf(m, mx);
    const float base = nm == -INFINITY ? 0.f : nm;
    const float corr = __builtin_amdgcn_exp2f(m - base);
    m = nm;
    s *= corr;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      x[i] = __builtin_amdgcn_exp2f(x[i] - base);
      s += x[i];
    }
    if (__any(corr != 1.f)) {
#pragma unroll
      for (int i = 0; i < VT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] *= corr;
    }
    // weights in three bf16 parts, whose sum they are; of bf16 pools none of them 0
    u32x4 w[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
      for (int i = 0; i < NK / 2; ++i) {
        const float lo = !FP8 && t < 2 ? next_below(x[i * 2]) : x[i * 2];
        const float hi = !FP8 && t < 2 ? next_below(x[i * 2 + 1]) : x[i * 2 + 1];
        w[t][i] = pack_hi(lo, hi);
        x[i * 2] -= high_half(lo);
        x[i * 2 + 1] -= high_half(hi);
      }
    }
    // Rows that are not the sequence's (behind its end in its last page, in front
    // of its window) may hold anything, and a weight of 0 does not undo a NaN
    const bool edge = np < PGS || c0 + PGS * BS > t1 || (EXT && c0 < wstart);
    wait(nn);
    if constexpr (NEW) {
      const int p = (last - c0) / BS, r = last % BS;
      if (own && lane < CPR)
        *reinterpret_cast<u32x4*>(vl + p * PAGE + r * RB +
                                  value_chunk(lane, p * BS + r) * 16) =
            *reinterpret_cast<const u32x4*>(new_kv[1] + lane * 16);
    }
    auto weigh = [&](auto masked) {
      u32x4 keep;
      if constexpr (masked.value) {
#pragma unroll
        for (int j = 0; j < NK / 2; ++j) {
          const int tok = c0 + (j >> 1) * 16 + g * 4 + (j & 1) * 2;
          auto ok = [&](int t) {
            return (j >> 1) < np && t < t1 && (!EXT || t >= wstart);
          };
          keep[j] = (ok(tok) ? 0x0000ffffu : 0) | (ok(tok + 1) ? 0xffff0000u : 0);
        }
      }
#pragma unroll
      for (int i = 0; i < VT; ++i) {
        u32x4 a;                             // keys g*4 .. of both pages
        if constexpr (FP8) {
          const int r = sub >> 1, row = (r >> 2) * BS + g * 4 + (r & 3);
          a = fp8x8_bf16(__builtin_bit_cast(
              u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
                         (__attribute__((address_space(3))) i32x2*)(
                             vl + row * RB + value_chunk(i, row) * 16 +
                             (sub & 1) * 8))));
        } else {
#pragma unroll
          for (int p = 0; p < PGS; ++p) {
            const int row = p * BS + g * 4 + (sub >> 2);
            const u32x2 t = __builtin_bit_cast(
                u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                           (__attribute__((address_space(3))) s16x4*)(
                               vl + row * RB +
                               value_chunk(i * 2 + ((sub >> 1) & 1), row) * 16 +
                               (sub & 1) * 8)));
            a[p * 2] = t[0];
            a[p * 2 + 1] = t[1];
          }
        }
        if constexpr (masked.value) a &= keep;
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          if constexpr (PGS == 2)
            acc[i] = mfma16(a, w[t], acc[i]);
          else
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(
                __builtin_bit_cast(s16x4, u32x2{a[0], a[1]}),
                __builtin_bit_cast(s16x4, u32x2{w[t][0], w[t][1]}), acc[i], 0, 0,
                0);
        }
      }
    };
    if (edge) weigh(std::true_type{});
    else weigh(std::false_type{});
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the values are read
    if (nn > 0) stage_v(next, nn);
    c0 = cn;
    np = nn;
    page[0] = next[0];
    page[1] = next[1];
  }

  if (nsplit > 1 && t0 >= len) return;     // the join skips it as well
  // the four key groups of a wave, then the waves
  s = sum_groups(s);
  float* sums = reinterpret_cast<float*>(kl);      // [GQ, OS], this wave's
  if (sub < GQ) {
#pragma unroll
    for (int i = 0; i < VT; ++i)
      *reinterpret_cast<f32x4*>(sums + sub * OS + i * 16 + g * 4) = acc[i];
    if (g == 0) {
      lds_ms[wave][sub][0] = m;
      lds_ms[wave][sub][1] = s;
    }
  }
  __syncthreads();

  for (int u = threadIdx.x; u < GQ * (D / 4); u += THREADS) {
    const int gq = u / (D / 4), d = u % (D / 4) * 4;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) M = fmaxf(M, lds_ms[w][gq][0]);
    float extra = 0.f;
    if constexpr (EXT) {
      // an attention sink joins the softmax denominator only; with several
      // parts the join adds it
      if (sinks != nullptr && whole) {
        const float sk = sinks[h * GQ + gq] * LOG2E;
        M = fmaxf(M, sk);
        extra = __builtin_amdgcn_exp2f(sk - M);
      }
    }
    const float base = M == -INFINITY ? 0.f : M;
    f32x4 num{0.f, 0.f, 0.f, 0.f};
    float den = extra;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
      const float wt = __builtin_amdgcn_exp2f(lds_ms[w][gq][0] - base);
      const f32x4 a = *reinterpret_cast<const f32x4*>(
          reinterpret_cast<const float*>(lds + w * RING) + gq * OS + d);
#pragma unroll
      for (int j = 0; j < 4; ++j) num[j] += wt * a[j];
      den += wt * lds_ms[w][gq][1];
    }
    if (whole) {
      u16x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = f2bf(den > 0.f ? num[j] / den : 0.f);
      *reinterpret_cast<u16x4*>(
          out + ((long)seq * Hq + (long)h * GQ + gq) * D + d) = o;
    } else {
      float* pp = part + ((((long)seq * Hkv + h) * nsplit + blockIdx.z) * GQ +
                          gq) * (D + 2);
#pragma unroll
      for (int j = 0; j < 4; ++j) pp[d + j] = num[j];
      if (d == 0) {
        pp[D] = M;
        pp[D + 1] = den;
      }
    }
  }
}

// Joins the parts of one (sequence, query head): a few KB that the decode
// kernel left in the L2, bound by the launch and two round trips, the length's and the
// parts', of which eight at a time are on their way.
template <int D>
__global__ __launch_bounds__(D) void paged_attn_join_kernel(
    unsigned short* __restrict__ out,       // [N, Hq, D]
    const float* __restrict__ part,         // [N, Hkv, nsplit, GQ, D + 2]
    const int* __restrict__ seq_lens, int GQ, int nsplit, int least,
    const float* __restrict__ sinks, int window) {
  constexpr int U = 8;
  const int seq = blockIdx.x, hq = blockIdx.y, Hq = gridDim.y;
  const int h = hq / GQ, gq = hq % GQ, d = threadIdx.x;
  const int len = seq_lens[seq];
  const int keys = len - window_start(len, window) / BS * BS;
  const int span = part_tokens(keys, nsplit, least);
  const int n = min(nsplit, (keys + span - 1) / span);
  if (n == 1) return;                      // the decode kernel's own result
  const float* pp = part +
      (((long)seq * (Hq / GQ) + h) * nsplit * GQ + gq) * (D + 2);
  const long step = (long)GQ * (D + 2);
  float M = -INFINITY, num = 0.f, den = 0.f;
  if (sinks != nullptr) {
    M = sinks[hq] * LOG2E;
    den = 1.f;
  }
  for (int i0 = 0; i0 < n; i0 += U) {
    float v[U], mx[U], dn[U], top = M;
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const float* at = pp + min(i0 + i, n - 1) * step;
      v[i] = at[d];
      mx[i] = at[D];
      dn[i] = at[D + 1];
    }
#pragma unroll
    for (int i = 0; i < U; ++i) top = fmaxf(top, mx[i]);   // the last one again
    const float base = top == -INFINITY ? 0.f : top;
    const float was = __builtin_amdgcn_exp2f(M - base);
    num *= was;
    den *= was;
    M = top;
#pragma unroll
    for (int i = 0; i < U; ++i)
      if (i0 + i < n) {
        const float wt = __builtin_amdgcn_exp2f(mx[i] - base);
        num += wt * v[i];
        den += wt * dn[i];
      }
  }
  out[((long)seq * Hq + hq) * D + d] = f2bf(den > 0.f ? num / den : 0.f);
}

}  // namespace

// Parts per sequence, and the fewest keys of one: parts fill the chip when
// sequences x kv heads (`base`) do not, but each writes its sums to memory and the
// join is a launch. max_blocks is the width of the block table, so a captured graph
// keeps its grid; parts behind a sequence's end return at once.
// Groups of heads: one workgroup a CU, whose waves keep 64 KB under way, brings 5.5
// TB/s, rows of 128 bytes (fp8, or 64 channels) want two and of 64 bytes four. Few more
// than one a CU leave most CUs idle beside those with two, and are cut; twice as many
// even out. us, 32 heads on 8 of 128 channels in bf16 unless said (parts chosen: time /
// others):
//   one sequence, 4500 keys   16: 14.9 / 8: 15.5, 1: 44; 4 x 2000 to 6000 8: 20.0 / 12: 20.1
//   8 x 1000 to 8000          4: 39.4 / 3: 40, 1: 76; 300 to 1200 4: 12.8 / 1: 15.3
//   12 x 3900                 2: 40.6 / 4: 44, 1: 48; 1000 to 8000 2: 54 / 16: 53, 1: 79
//   16 x 1000 to 8000         2: 69 / 4: 71, 1: 84; 300 to 1200 2: 16.1 / 1: 16.4, 4: 16.9
//   24 x 1000 to 8000         1: 95 / 4: 102; all of 500 1: 12.9 / 2: 14.2
//   17 x 2600                 1: 37 / 3: 41; 300 to 1200 1: 17 / 4: 19; 1000 to 6000 1: 68 / 16: 57
//   32 x 1000 to 8000         1: 119 / 3: 126; 34 x 2600 4: 74 / 1: 79; 1000 to 6000 4: 104 / 1: 131
//   44 x 2600                 3: 91 / 1: 91; 1000 to 6000 3: 134 / 1: 149; 56 x 1: 170 / 4: 171
//   64 channels in fp8: 24 x 1000 to 6000 5: 29 / 1: 57; 48 x 2: 47 / 1: 64; 64 x 1: 67 / 2: 62
//   256 channels: 37 x 2600   4: 151 / 1: 168; 1000 to 6000 4: 209 / 1: 275; 48 x 3: 296 / 1: 313
//   fp8: 8 x 1000 to 8000     8: 25.9 / 4: 27; 16 x 4: 41 / 6: 42; 24 x 2: 57 / 4: 56, 1: 75
//        32 x 1000 to 8000    1: 81 / 2: 71, all of 3900 1: 47 / 2: 53; 300 to 1200 1: 16.2 / 2: 17.4
// Single heads, whose workgroups bring less each, are cut for twice as many, narrow rows
// for four times, and heads of 256 channels, of which few workgroups fit at once, too,
// but not into more than 8 parts.
// A context of less than one part pays for the join's launch behind a wide
// block table (one sequence of 100 keys, 8 heads on 8: 5.8 against 4.4).
// Up to 64 groups (128 of 64-byte rows) parts of 128 keys, one step, where the table has
// more than 256 and the join is there anyway, one part up to there. us, parts of 256 / of
// 128, 16 heads on 8: 3 x 200 to 400 7.8 / 6.5, 8 7.9 / 7.0, 3 x 500 to 1200 8.3 / 7.4, 8
// 10.7 / 10.7, 6 9.1 / 9.5; of 256 channels 3 x 200 to 400 .78 of the time, in fp8 .81; but
// behind a table of 200 3 x 128 to 200 in one part 5.0, in two 6.2.
// Two heads a kv head of 64 channels go through paged_attn_heads_kernel as a pair in fp8,
// and in bf16 behind tables of up to 64 keys up to 512 groups (256 groups .87 of the time,
// 768 1.06).
// aligned: the pools take 16-byte direct loads.
DecodeParts decode_parts(int N, int Hq, int Hkv, int max_blocks, int D, int fp8,
                         int window, int aligned) {
  const bool grouped = Hq > Hkv && aligned && max_blocks > 0;
  const bool pairs =
      grouped && Hq == 2 * Hkv && D == 64 &&
      (fp8 || (max_blocks <= 4 && (long)N * Hkv <= 512));
  const int heads = pairs ? 2 : grouped ? 0 : 1;
  const long base = (long)N * (grouped ? Hkv : Hq);
  if (base < 1) return {1, 4 * STEP, heads};
  long keys = (long)max_blocks * BS;
  if (window > 0 && window < keys) keys = window;
  const bool narrow = D * (fp8 ? 1 : 2) <= 128;
  long n, cap = 16;
  int least;
  if (heads == 0) {
    const int row = D * (fp8 ? 1 : 2);
    n = row <= 64     ? (base >= 512 ? 1 : 1024 / base)
        : row <= 128  ? (base >= 256 ? 1 : 512 / base)
        : base <= 256 ? 256 / base
        : base < 400  ? (1024 + base - 1) / base
                      : 1;
    least = base > (row <= 64 ? 128 : 64) ? 512 : keys > 256 ? 128 : 256;
  } else {
    n = narrow        ? (pairs && base >= 512 ? 1 : 1024 / base)
        : base >= 512 ? 1
        : D > 128     ? (1024 + base - 1) / base
                      : (512 + base - 1) / base;
    least = base >= 256 ? 512 : base >= 128 ? 256 : 128;
    if (D > 128) cap = 8;
  }
  const long most =
      base >= 128 && heads > 0 ? keys / least : (keys + least - 1) / least;
  if (n > most) n = most;
  return {(int)(n < 1 ? 1 : n > cap ? cap : n), least, heads};
}

namespace {
struct DecodeArgs {
  unsigned short* out;
  const unsigned short* q;
  const char *kc, *vc;
  const int *block_tables, *seq_lens;
  float* part;
  DecodeParts parts;
  int N, Hq, Hkv, max_blocks;
  float scale;
  long q_stride;
  const float* sinks;
  int window;
  float softcap;
  NewRows rows;             // or none of it, slots null
  hipStream_t s;
};

template <int D, bool FP8, bool EXT>
void decode_launch(const DecodeArgs& a) {
  const int GQ = a.Hq / a.Hkv;
  auto run = [&](auto kernel, int units, int per, auto... extra) {
    hipLaunchKernelGGL(kernel, dim3(a.N, units, a.parts.n), dim3(THREADS), 0, a.s,
                       a.out, a.q, a.kc, a.vc, a.block_tables, a.seq_lens, a.part,
                       a.parts.least, a.Hkv, per, a.max_blocks, a.scale, a.q_stride,
                       a.sinks, a.window, a.softcap, extra...);
  };
  if (a.parts.heads == 1) {
    run(paged_attn_heads_kernel<D, 1, FP8, EXT>, a.Hq, GQ);
    return;
  }
  if constexpr (D == 64) {
    if (a.parts.heads == 2) {
      run(paged_attn_heads_kernel<D, 2, FP8, EXT>, a.Hkv, 1);
      return;
    }
  }
  // Pages a step: two of fp8 rows, one of 256 channels in bf16; of fewer in bf16 two up to
  // one workgroup a CU, which then has more under way (us, one page / two: 32 sequences of
  // 1000 to 6000 keys, 32 heads on 8 of 128 99 / 93, 24 of 300 to 1200 21.4 / 19.0, but of
  // 40 to 60 4.4 / 4.8), one where they are more and share it (40 x 300 to 1200 32.1 /
  // 34.4, 64 x 500 29.5 / 33.0, 512 x 40 to 60 26.1 / 33.9, but 384 x 200 to 400 93 / 88; of
  // 64 channels, 16 heads on 8, five of whose workgroups then share it, 384 x 20 to 64
  // 10.0 / 12.9, 128 x 200 to 400 .94 to 1.02, 500 to 1200 .96 to .99 of the time).
  constexpr bool ONE = !FP8, TWO = FP8 || D <= 128;
  constexpr bool FUSED = D == 128 && !EXT;
  if constexpr (ONE) {
    if (!TWO || (long)a.N * a.Hkv > 256) {
      if (FUSED && a.rows.slots != nullptr)
        run(paged_attn_decode_kernel<D, FP8, EXT, 1, FUSED>, a.Hkv, GQ, a.rows);
      else
        run(paged_attn_decode_kernel<D, FP8, EXT, 1, false>, a.Hkv, GQ, a.rows);
      return;
    }
  }
  if constexpr (TWO) {
    if (FUSED && a.rows.slots != nullptr)
      run(paged_attn_decode_kernel<D, FP8, EXT, 2, FUSED>, a.Hkv, GQ, a.rows);
    else
      run(paged_attn_decode_kernel<D, FP8, EXT, 2, false>, a.Hkv, GQ, a.rows);
  }
}
}  // namespace

// rows: where q is null, the step's own (heads of 128 channels, several of them a kv head,
// no option); every sequence has one row.
void paged_attn_decode_launch(void* out, const void* q, const void* kc,
                              const void* vc, const int* block_tables,
                              const int* seq_lens, float* part, DecodeParts parts,
                              int N, int Hq, int Hkv, int D, int max_blocks,
                              float scale, long q_stride, int fp8,
                              const float* sinks, int window, float softcap,
                              const NewRows* rows, int* err_unsupported,
                              hipStream_t s) {
  const int GQ = Hq / Hkv, nsplit = parts.n;
  const bool ext = (sinks != nullptr) || window > 0 || softcap > 0.f;
  *err_unsupported = (D != 128 && D != 64 && D != 256) || GQ < 1 || GQ > 8 ||
                     GQ == 3 || (D == 256 && GQ > 4) ||
                     (rows != nullptr && (D != 128 || ext || parts.heads != 0));
  if (*err_unsupported || N == 0) return;
  const DecodeArgs a{(unsigned short*)out, (const unsigned short*)q,
                     (const char*)kc, (const char*)vc, block_tables, seq_lens,
                     part, parts, N, Hq, Hkv, max_blocks, scale, q_stride, sinks,
                     window, softcap, rows != nullptr ? *rows : NewRows{}, s};
  if (D == 128 && !ext) (fp8 ? decode_launch<128, true, false> : decode_launch<128, false, false>)(a);
  else if (D == 128) (fp8 ? decode_launch<128, true, true> : decode_launch<128, false, true>)(a);
  else if (D == 64) (fp8 ? decode_launch<64, true, true> : decode_launch<64, false, true>)(a);
  else (fp8 ? decode_launch<256, true, true> : decode_launch<256, false, true>)(a);
  if (nsplit <= 1) return;
#define JOIN(DD)                                                              \
  hipLaunchKernelGGL((paged_attn_join_kernel<DD>), dim3(N, Hq), dim3(DD), 0,  \
                     s, (unsigned short*)out, part, seq_lens,                 \
                     parts.heads == 0 ? GQ : parts.heads, nsplit,             \
                     parts.least, sinks, window)
  if (D == 128) JOIN(128);
  else if (D == 64) JOIN(64);
  else JOIN(256);
#undef JOIN
}
