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
//  - 4 waves per workgroup, 32 keys (two pages) per wave and step; the last
//    step, and the only one of parts of up to 64 keys, may be of one page (us,
//    8 heads on 8: 64 x 400 keys in a window of 128 9.5 -> 7.1, 512 x 40 20.1 ->
//    18.2 and in fp8 18.7 -> 16.5). Scores are
//    a matrix product, S^T = K Q^T on mfma_f32_16x16x32_bf16: K rows are the
//    16-byte loads of the A operand as they lie in the page, the GQ query
//    rows (zero rows up to 16) the B operand. One lane then holds one head's
//    scores of 8 keys, so maximum and sum take two cross-lane steps per 32
//    keys instead of four per key.
//  - probabilities stay fp32: they go through LDS to a layout of 16 lanes a
//    value row (D/16 channels each) x 4 keys, where the weighted sum is fp32
//    FMA on values loaded 16 bytes (bf16) or 8 bytes (fp8) a lane.
//  - fp8 keys become bf16 exactly (e4m3 has 3 mantissa bits) in registers.
//
// Bound by the K/V stream: 32 keys cost a SIMD about 1300 cycles (GQ = 4),
// 31 TB/s over the chip in bf16 and 15 TB/s in fp8, so memory sets the time
// once enough of it is in flight (16 KB a wave in bf16 at 128 channels;
// decode_waves has the waves a SIMD).
//
// KV pool layout: [num_blocks, Hkv, BS, D] bf16 | fp8, BS = 16 tokens.
#include "common.h"

#include <type_traits>

struct DecodeParts { int n, least; };   // of a sequence, and a part's keys

namespace {

constexpr int BS = 16;       // tokens per KV block (page)
constexpr int NWAVES = 4;    // waves per workgroup
constexpr int THREADS = NWAVES * WAVE_SIZE;
constexpr int STEP = 32;     // keys per wave and step (two pages)
constexpr float LOG2E = 1.4426950408889634f;

typedef __attribute__((ext_vector_type(8))) short s16x8;
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

// A value and the one of the lane 16 or 32 away, in either order, without the
// LDS: as shuffles these exchanges, most of them in the sums at the end, were
// 12 % of the kernel over 240 shapes (16 heads of 256, us: 512 x 40 keys
// 53.6 -> 42.0, one x 300 12.2 -> 11.1; 32 of 128: 64 x 400 21.0 -> 19.2). The two
// operands are kept apart, as in half_wave_max.
template <int M>
DEVICE_INLINE f32x2 with_lane(float v) {
  const unsigned int a = __builtin_bit_cast(unsigned int, v);
  unsigned int b = a;
  asm("" : "+v"(b));
  const auto r = M == 16 ? __builtin_amdgcn_permlane16_swap(a, b, false, false)
                         : __builtin_amdgcn_permlane32_swap(a, b, false, false);
  const unsigned int x = r[0], y = r[1];
  return f32x2{__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
}
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

// Waves that a SIMD holds beside each other. Left to itself the compiler takes
// a few registers too many for four of them at 4 heads in fp8 and for three at
// 8 in bf16 (us: 256 x 400 keys 43 -> 49, 93 -> 99).
constexpr int decode_waves(int D, int GQ, bool fp8) {
  return D == 64    ? (GQ <= 6 ? 5 : 4)
         : D == 256 ? (fp8 && GQ <= 2 ? 3 : 2)
                    : (GQ <= 2 || (fp8 && GQ <= 5) ? 4 : 3);
}

// EXT: sinks / sliding window / softcap (GPT-OSS and Gemma variants).
template <int D, int GQ, bool FP8, bool EXT>
__global__ __launch_bounds__(THREADS, decode_waves(D, GQ, FP8))
void paged_attn_decode_kernel(
    unsigned short* __restrict__ out,        // [N, Hq, D]
    const unsigned short* __restrict__ q,    // [N, Hq, D]
    const void* __restrict__ kc,             // [B, Hkv, BS, D] bf16|fp8
    const void* __restrict__ vc,             // [B, Hkv, BS, D]
    const int* __restrict__ block_tables,    // [N, max_blocks]
    const int* __restrict__ seq_lens,        // [N]
    float* __restrict__ part,                // [N, Hkv, nsplit, GQ, D + 2]
    int least,                               // keys of a part (part_tokens)
    int Hkv, int max_blocks, float scale, long q_stride,
    const float* __restrict__ sinks,         // [Hq] or null (GPT-OSS)
    int window,                              // 0 = full attention
    float softcap) {                         // 0 = off (Gemma-2 tanh cap)
  constexpr int DV = D / 16;        // value channels per lane
  constexpr int ES = FP8 ? 1 : 2;   // bytes per cached number
  constexpr int QK = D / 32;        // products per 16 keys
  constexpr int KW = 8 * ES / 4;    // words of a K fragment
  constexpr int VW = DV * ES / 4;   // words of a lane's value channels
  constexpr int GP = GQ <= 2 ? GQ : (GQ + 3) / 4 * 4;  // padded P row
  static_assert(D == 64 || D == 128 || D == 256, "D in {64, 128, 256}");

  const int seq = blockIdx.x;
  const int h = blockIdx.y;         // kv head
  const int nsplit = gridDim.z;
  const int Hq = Hkv * GQ;
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

  __shared__ float lds_p[NWAVES][STEP][GP];
  __shared__ float lds_c[NWAVES][GP];
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

  const char* kbase = reinterpret_cast<const char*>(kc) + (long)h * BS * D * ES;
  const char* vbase = reinterpret_cast<const char*>(vc) + (long)h * BS * D * ES;
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
      float* pp = part + ((((long)seq * Hkv + h) * nsplit + blockIdx.z) * GQ +
                          gq) * (D + 2);
      pp[d] = num;
      if (d == 0) {
        pp[D] = M;
        pp[D + 1] = den;
      }
    }
  }
}

// Joins the parts of one (sequence, query head): a few KB that the decode
// kernel left in the L2, bound by the launch.
template <int D>
__global__ __launch_bounds__(D) void paged_attn_join_kernel(
    unsigned short* __restrict__ out,       // [N, Hq, D]
    const float* __restrict__ part,         // [N, Hkv, nsplit, GQ, D + 2]
    const int* __restrict__ seq_lens, int GQ, int nsplit, int least,
    const float* __restrict__ sinks, int window) {
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
  float M = -INFINITY;
  for (int i = 0; i < n; ++i) M = fmaxf(M, pp[i * step + D]);
  float num = 0.f, den = 0.f;
  if (sinks != nullptr) {
    const float sk = sinks[hq] * LOG2E;
    M = fmaxf(M, sk);
    den = __builtin_amdgcn_exp2f(sk - M);
  }
  const float base = M == -INFINITY ? 0.f : M;
  for (int i = 0; i < n; ++i) {
    const float wt = __builtin_amdgcn_exp2f(pp[i * step + D] - base);
    num += wt * pp[i * step + d];
    den += wt * pp[i * step + D + 1];
  }
  out[((long)seq * Hq + hq) * D + d] = f2bf(den > 0.f ? num / den : 0.f);
}

}  // namespace

// Parts per sequence, and the fewest keys of one: parts fill the chip when
// sequences x kv heads (`base`) do not, and even out unequal lengths, but each
// writes its sums to memory and the join is a launch. max_blocks is the width
// of the block table, so a captured graph keeps its grid; parts behind a
// sequence's end return at once. Measured with 1 to 32 parts, us, 32 heads on
// 8 of 128 channels in bf16 unless said (parts chosen: time / others):
//   one sequence, 4000 keys   16: 17 / 8: 16.5, 32: 23, 1: 49
//   8, 200 to 8000            8: 37 / 4: 39, 32: 48, 1: 112
//   16, 1000 to 8000          4: 66 / 1: 137, 16: 71; 300 to 1200 2: 18 / 1: 22
//   32, 1000 to 8000          2: 134 / 1: 154, 8: 140; all of 300: 2: 12.5 / 1: 10.9
//   48, 3500 to 7900          2: 219 / 1: 237, 6: 225; 100 to 600 2: 21 / 1: 19
//   64, 100 to 4000           1: 125 / 2: 134, 4: 131; all of 300: 1: 16.7 / 4: 18.9
// Rows of 128 bytes (fp8, or 64 channels) spend relatively more on scores, so
// they are cut for twice as many workgroups:
//   fp8: 64, 100 to 4000      2: 86 / 1: 83, 4: 82; 32, 1000 to 8000 4: 90 / 1: 141, 2: 97
//        96, 100 to 4000      1: 117 / 2: 132; 48, 3500 to 7900 2: 131 / 1: 179, 4: 150
// So are heads of 256 channels, of which few workgroups fit at once, but not
// into more than 8 parts (16 heads on 8):
//        48, 3500 to 7900     3: 436 / 1: 486, 6: 414; 24, 200 to 2000 6: 48 / 1: 51
//        64, 100 to 4000      1: 240 / 4: 247, 8: 259
// A context of less than one part pays for the join's launch behind a wide
// block table (one sequence of 100 keys, 8 heads on 8: 5.8 against 4.4).
DecodeParts decode_parts(int N, int Hkv, int max_blocks, int D, int fp8,
                         int window) {
  const long base = (long)N * Hkv;
  if (base < 1) return {1, 4 * STEP};
  const bool narrow = D * (fp8 ? 1 : 2) <= 128;
  long n = narrow    ? 1024 / base
           : base >= 512 ? 1
           : D > 128     ? (1024 + base - 1) / base
                         : (512 + base - 1) / base;
  const int least = base >= 256 ? 512 : base >= 128 ? 256 : 128;
  long keys = (long)max_blocks * BS;
  if (window > 0 && window < keys) keys = window;
  const long most = base >= 128 ? keys / least : (keys + least - 1) / least;
  if (n > most) n = most;
  const long cap = D > 128 ? 8 : 16;
  return {(int)(n < 1 ? 1 : n > cap ? cap : n), least};
}

void paged_attn_decode_launch(void* out, const void* q, const void* kc,
                              const void* vc, const int* block_tables,
                              const int* seq_lens, float* part, DecodeParts parts,
                              int N, int Hq, int Hkv, int D, int max_blocks,
                              float scale, long q_stride, int fp8,
                              const float* sinks, int window, float softcap,
                              int* err_unsupported, hipStream_t s) {
  const int GQ = Hq / Hkv, nsplit = parts.n;
  dim3 grid(N, Hkv, nsplit);
  dim3 block(THREADS);
  *err_unsupported = 0;
  if (D != 128 && D != 64 && D != 256) { *err_unsupported = 1; return; }
  if (D == 256 && GQ > 4) { *err_unsupported = 1; return; }  // VGPR budget
  const bool ext = (sinks != nullptr) || window > 0 || softcap > 0.f;
#define LAUNCH_D(DD, G, F, E)                                                  \
  hipLaunchKernelGGL((paged_attn_decode_kernel<DD, G, F, E>), grid, block, 0,  \
                     s, (unsigned short*)out, (const unsigned short*)q, kc,    \
                     vc, block_tables, seq_lens, part, parts.least, Hkv,       \
                     max_blocks, scale, q_stride, sinks, window, softcap)
#define LAUNCH_GQ2(G, F)                                                       \
  do {                                                                         \
    if (D == 128) {                                                            \
      if (ext) LAUNCH_D(128, G, F, true);                                      \
      else LAUNCH_D(128, G, F, false);                                         \
    } else if (D == 64) {                                                      \
      LAUNCH_D(64, G, F, true);                                                \
    } else if ((G) <= 4) {                                                     \
      LAUNCH_D(256, (G) <= 4 ? (G) : 1, F, true);                              \
    }                                                                          \
  } while (0)
#define LAUNCH_GQ(G)                                                          \
  do {                                                                        \
    if (fp8) LAUNCH_GQ2(G, true);                                             \
    else LAUNCH_GQ2(G, false);                                                \
  } while (0)
  switch (GQ) {
    case 1: LAUNCH_GQ(1); break;
    case 2: LAUNCH_GQ(2); break;
    case 4: LAUNCH_GQ(4); break;
    case 5: LAUNCH_GQ(5); break;
    case 6: LAUNCH_GQ(6); break;
    case 7: LAUNCH_GQ(7); break;
    case 8: LAUNCH_GQ(8); break;
    default: *err_unsupported = 1; return;
  }
#undef LAUNCH_GQ
#undef LAUNCH_GQ2
#undef LAUNCH_D
  if (nsplit <= 1) return;
#define JOIN(DD)                                                              \
  hipLaunchKernelGGL((paged_attn_join_kernel<DD>), dim3(N, Hq), dim3(DD), 0,  \
                     s, (unsigned short*)out, part, seq_lens, GQ, nsplit,     \
                     parts.least, sinks, window)
  if (D == 128) JOIN(128);
  else if (D == 64) JOIN(64);
  else JOIN(256);
#undef JOIN
}
