// Paged rotary attention over a ragged batch (gfx950).
//
//   out[t, a, :] = sum_j softmax_j(scale * q[t, a, :] . k_j) * v_j
//
// over the visible keys j of row t's sequence, read through its block
// table: j <= pos(t), and with a window also (pos(t) - j < window or
// j < keep_first), or, in chunks, only keys of the row's own chunk of
// positions, j >= pos(t) - pos(t) mod chunk. a runs over heads * maps SCORE MAPS (a = head * maps +
// map): map m of a head reads channels [m*D, (m+1)*D) of its kv head's key
// row, and all maps of a head weight the same value rows — two maps per
// head are the two halves of differential attention, combined afterwards.
// A per-head sink logit may join the denominator (no key, no value), and a
// per-head slope times the distance pos(t) - j may be taken off the scaled
// score (positions without rotation); a tanh cap may bound the scaled
// score; a sigmoid gate per row and head may multiply the output. q and out
// are [T, A, *] views with a contiguous last axis.
//
// Pools: keys [nblocks, G, BS, KW] with KW = maps * D (rotated at write
// time), values with every page transposed, [nblocks, G, VW, BS], so both
// matrix products find their reduction axis contiguous: scores reduce over
// channels, the weighted sum over keys.
//
// A workgroup takes a tile of up to 16 (row, map) pairs that share one key
// stream — same sequence, same kv head, same map (host-built list: 16 rows
// x 1 map inside prompts, rows x the query heads of a kv group for decode
// rows) — and walks that stream once for all of them. Each pair sees the
// keys from a lower bound of its own up to its position, plus the kept first
// keys; the walk visits the key tiles of the kept keys and those from the
// pairs' smallest bound on, so a windowed or chunked layer costs its window
// or chunk, not its context.
//
// Two paths. The MFMA path (bf16 q and pools, BS = 16, D % 32 == 0, VW %
// 16 == 0) runs both products on v_mfma_f32_16x16x32_bf16 with fp32
// accumulation; scores are scaled, masked and soft-maxed in fp32 and only
// the weights are rounded to bf16 for the second product. Per 64-key tile:
// wave w multiplies the 16 pairs with keys 16w..16w+15 (B operand straight
// from the key pool, 16 B per lane), scores meet in LDS for the online
// softmax, then wave w owns the output channels of n-tiles w, w+4, ... and
// multiplies P (A operand, LDS) with the transposed value pages; heads of 128
// channels have a kernel of their own (paged_attn_waves_kernel). With few
// tiles over long contexts (decode) gridDim.y workgroups split a tile's
// keys and a merge kernel joins the partial (acc, m, l) triples. The exact
// path keeps everything fp32 on the vector ALUs, for pools of bf16 or fp32
// and any sizes; it is the path of fp32 engines and the reference the MFMA
// kernel is tested against.
#include "common.h"

#include <type_traits>

namespace {

constexpr int G16 = 16;       // (row, map) pairs per workgroup
constexpr int THREADS = 256;

template <typename T> DEVICE_INLINE float ldf(const T* p);
template <> DEVICE_INLINE float ldf<float>(const float* p) { return *p; }
template <> DEVICE_INLINE float ldf<unsigned short>(const unsigned short* p) {
  return bf2f(*p);
}
template <typename T> DEVICE_INLINE void stf(T* p, float v);
template <> DEVICE_INLINE void stf<float>(float* p, float v) { *p = v; }
template <> DEVICE_INLINE void stf<unsigned short>(unsigned short* p, float v) {
  *p = f2bf(v);
}

struct AttnArgs {
  const int* block_tables;   // [nseq, maxb]
  const int* tiles;          // [ntiles, 6] row0, nrows, a0, n_a, seq, a_step
  const int* pos32;          // [T]
  const float* sinks;        // [A / maps] or null
  const float* slopes;       // [A / maps] or null
  float scale;
  float softcap;             // > 0: scaled scores pass cap * tanh(s / cap)
  long q_st, q_sa;           // element strides of q [T, A, D]: row, score map
  long o_st, o_sa;           // and of out [T, A, VW]
  int T, A, D, VW, KW, G, BS, maps, rep;   // rep = heads / kv heads
  int nseq, maxb, nblocks, window, keep_first, chunk;
  const void* gate;          // [T, A / maps] view in q's dtype, or null
  long g_st;
};

// Decodes and validates a tile; false = skip the tile untouched.
DEVICE_INLINE bool tile_setup(const AttnArgs& p, int tile, int* e_pos,
                              int* e_lo, int* e_row, int* e_a, int& n_ent,
                              int& seq, int& g, int& koff) {
  const int* tl = p.tiles + (long)tile * 6;
  const int row0 = tl[0], nrows = tl[1], a0 = tl[2], n_a = tl[3];
  const int a_step = tl[5];
  seq = tl[4];
  if (row0 < 0 || nrows < 1 || row0 + nrows > p.T || a0 < 0 || n_a < 1 ||
      a_step < 1 || a0 + (long)(n_a - 1) * a_step >= p.A ||
      (long)nrows * n_a > G16 || seq < 0 || seq >= p.nseq)
    return false;
  n_ent = nrows * n_a;
  g = (a0 / p.maps) / p.rep;
  koff = (a0 % p.maps) * p.D;
  if (g >= p.G) return false;
  if (threadIdx.x < G16) {
    int ps = -1, lo = 1 << 30, row = 0, a = 0;
    if ((int)threadIdx.x < n_ent) {
      row = row0 + threadIdx.x / n_a;
      a = a0 + (threadIdx.x % n_a) * a_step;
      ps = min(max(p.pos32[row], 0), p.maxb * p.BS - 1);
      lo = p.window > 0 ? max(0, ps - p.window + 1) : 0;
      if (p.chunk > 0) lo = max(lo, ps - ps % p.chunk);
    }
    e_pos[threadIdx.x] = ps;
    e_lo[threadIdx.x] = lo;
    e_row[threadIdx.x] = row;
    e_a[threadIdx.x] = a;
  }
  return true;
}

DEVICE_INLINE bool key_visible(int j, int pos, int lo, int keep_first) {
  return j <= pos && (j >= lo || j < keep_first);
}

// The key tiles of KT keys a tile of pairs visits: those of the kept first
// keys, [0, kept), then [from, end). Position v of the walk is tile
// v < kept ? v : v - kept + from, v in [0, n).
struct KeyWalk {
  int kept, from, n;
  DEVICE_INLINE int tile(int v) const { return v < kept ? v : v - kept + from; }
};

DEVICE_INLINE KeyWalk key_walk(int lo, int jmax, int keep_first, int KT) {
  KeyWalk w;
  const int end = jmax / KT + 1;
  w.from = lo / KT;
  w.kept = min((keep_first + KT - 1) / KT, w.from);
  w.n = w.kept + end - w.from;
  return w;
}

template <typename TG>
DEVICE_INLINE float head_gate_of(const AttnArgs& p, int row, int a) {
  if (p.gate == nullptr) return 1.f;
  const float z = ldf((const TG*)p.gate + (long)row * p.g_st + a / p.maps);
  return 1.0f / (1.0f + expf(-z));
}

DEVICE_INLINE float scaled_score(float dot, const AttnArgs& p) {
  const float s = dot * p.scale;
  return p.softcap > 0.f ? p.softcap * tanhf(s / p.softcap) : s;
}

// ---- exact path ----------------------------------------------------------

template <typename TQ, typename TC, typename TO, int NJ, int KT>
__global__ __launch_bounds__(THREADS) void paged_attn_exact_kernel(
    TO* __restrict__ out, const TQ* __restrict__ q,
    const TC* __restrict__ k_cache, const TC* __restrict__ v_cache,
    AttnArgs p) {
  extern __shared__ float sm[];
  const int D = p.D, VW = p.VW, KS = p.D + 1, VS = p.VW + 1;
  float* qs = sm;                     // [16][D]
  float* ks = qs + G16 * D;           // [KT][KS]
  float* vs = ks + KT * KS;           // [KT][VS]
  float* ps = vs + KT * VS;           // [16][KT]
  float* als = ps + G16 * KT;         // [16]
  float* lsum = als + G16;            // [16]
  __shared__ int e_pos[G16], e_lo[G16], e_row[G16], e_a[G16];

  int n_ent, seq, g, koff;
  if (!tile_setup(p, blockIdx.x, e_pos, e_lo, e_row, e_a, n_ent, seq, g, koff))
    return;
  __syncthreads();
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int jmax = -1, lo = 1 << 30;
#pragma unroll
  for (int e = 0; e < G16; ++e) {
    jmax = max(jmax, e_pos[e]);
    lo = min(lo, e_lo[e]);
  }
  for (int e = wave; e < G16; e += 4) {
    const bool ok = e < n_ent;
    const TQ* qp = q + (long)e_row[e] * p.q_st + (long)e_a[e] * p.q_sa;
    for (int r = lane; r < D; r += 64) qs[e * D + r] = ok ? ldf(qp + r) : 0.f;
  }
  const int e_s = tid >> 4, kk = tid & 15;
  const int my_pos = e_pos[e_s], my_lo = e_lo[e_s];
  float m_run = -INFINITY, l_run = 0.f;
  if (p.sinks != nullptr && my_pos >= 0) {
    m_run = p.sinks[e_a[e_s] / p.maps];
    l_run = 1.f;
  }
  const float slope = p.slopes != nullptr ? p.slopes[e_a[e_s] / p.maps] : 0.f;
  float acc[4][NJ];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = 0.f;

  const int* bt = p.block_tables + (long)seq * p.maxb;
  const int BS = p.BS;
  const KeyWalk walk = key_walk(lo, jmax, p.keep_first, KT);
  for (int v = 0; v < walk.n; ++v) {
    const int k0 = walk.tile(v) * KT;
    __syncthreads();   // previous tile fully consumed (and qs written)
    for (int k = wave; k < KT; k += 4) {
      const int j = k0 + k;
      float* dst = ks + k * KS;
      if (j <= jmax) {
        const long blk = min(max(bt[j / BS], 0), p.nblocks - 1);
        const TC* src =
            k_cache + ((blk * p.G + g) * BS + j % BS) * (long)p.KW + koff;
        for (int r = lane; r < D; r += 64) dst[r] = ldf(src + r);
      } else {
        for (int r = lane; r < D; r += 64) dst[r] = 0.f;
      }
    }
    for (int i = tid; i < KT * VW; i += THREADS) {
      const int k = i % KT, c = i / KT;
      const int j = k0 + k;
      float v = 0.f;
      if (j <= jmax) {
        const long blk = min(max(bt[j / BS], 0), p.nblocks - 1);
        v = ldf(v_cache + ((blk * p.G + g) * (long)VW + c) * BS + j % BS);
      }
      vs[k * VS + c] = v;
    }
    __syncthreads();
    float s[KT / 16];
#pragma unroll
    for (int u = 0; u < KT / 16; ++u) s[u] = 0.f;
    {
      const float* qp = qs + e_s * D;
      for (int r = 0; r < D; ++r) {
        const float qv = qp[r];
#pragma unroll
        for (int u = 0; u < KT / 16; ++u) s[u] += qv * ks[(kk + 16 * u) * KS + r];
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < KT / 16; ++u) {
      const int j = k0 + kk + 16 * u;
      s[u] = key_visible(j, my_pos, my_lo, p.keep_first)
                 ? scaled_score(s[u], p) - slope * (float)(my_pos - j)
                 : -INFINITY;
      mx = fmaxf(mx, s[u]);
    }
#pragma unroll
    for (int m = 8; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, WAVE_SIZE));
    const float m_new = fmaxf(m_run, mx);
    float alpha = 1.f, psum = 0.f;
    if (m_new == -INFINITY) {
#pragma unroll
      for (int u = 0; u < KT / 16; ++u) ps[e_s * KT + kk + 16 * u] = 0.f;
    } else {
      alpha = expf(m_run - m_new);
#pragma unroll
      for (int u = 0; u < KT / 16; ++u) {
        const float pv = expf(s[u] - m_new);
        ps[e_s * KT + kk + 16 * u] = pv;
        psum += pv;
      }
    }
    psum = group16_reduce_sum(psum);
    l_run = l_run * alpha + psum;
    m_run = m_new;
    if (kk == 0) als[e_s] = alpha;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float al = als[wave + 4 * i];
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] *= al;
    }
    for (int k = 0; k < KT; ++k) {
      float vv[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int c = lane + 64 * j;
        vv[j] = c < VW ? vs[k * VS + c] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pv = ps[(wave + 4 * i) * KT + k];
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] += pv * vv[j];
      }
    }
  }
  if (kk == 0) lsum[e_s] = l_run;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = wave + 4 * i;
    if (e >= n_ent) continue;
    const float l = lsum[e];
    const float inv = (l > 0.f ? 1.0f / l : 0.f) *
                      head_gate_of<TQ>(p, e_row[e], e_a[e]);
    TO* op = out + (long)e_row[e] * p.o_st + (long)e_a[e] * p.o_sa;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int c = lane + 64 * j;
      if (c < VW) stf(op + c, acc[i][j] * inv);
    }
  }
}

// ---- MFMA path -------------------------------------------------------------

typedef __attribute__((ext_vector_type(8))) short ra_s16x8;

DEVICE_INLINE f32x4 ra_mfma(u16x8 a, u16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(ra_s16x8, a), __builtin_bit_cast(ra_s16x8, b), c, 0, 0, 0);
}

constexpr int MKT = 64;            // keys per tile (16 per wave)
constexpr int MSS = MKT + 4;       // fp32 score row stride
constexpr int MPS = MKT + 8;       // bf16 weight row stride (16 B aligned)

// NT: 16-channel n-tiles per wave (wave w owns n-tiles w, w+4, ...).
template <int NT, typename TO>
__global__ __launch_bounds__(THREADS) void paged_attn_mfma_kernel(
    TO* __restrict__ out, const unsigned short* __restrict__ q,
    const unsigned short* __restrict__ k_cache,
    const unsigned short* __restrict__ v_cache, AttnArgs p,
    float* __restrict__ ws_acc, float* __restrict__ ws_ml) {
  constexpr int BS = 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int D = p.D, VW = p.VW;
  const int QS = D + 8;                               // bf16 row stride
  unsigned short* Ql = reinterpret_cast<unsigned short*>(smem_raw);  // [16][QS]
  unsigned short* Pl = Ql + G16 * QS;                 // [16][MPS]
  float* Ss = reinterpret_cast<float*>(Pl + G16 * MPS);  // [16][MSS]
  float* als = Ss + G16 * MSS;                        // [16]
  float* lsum = als + G16;                            // [16]
  __shared__ int e_pos[G16], e_lo[G16], e_row[G16], e_a[G16];

  int n_ent, seq, g, koff;
  if (!tile_setup(p, blockIdx.x, e_pos, e_lo, e_row, e_a, n_ent, seq, g, koff))
    return;
  __syncthreads();
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lc = lane & 15, lg = lane >> 4;
  int jmax = -1, lo = 1 << 30;
#pragma unroll
  for (int e = 0; e < G16; ++e) {
    jmax = max(jmax, e_pos[e]);
    lo = min(lo, e_lo[e]);
  }
  for (int e = wave; e < G16; e += 4) {
    const bool ok = e < n_ent;
    const unsigned short* qp =
        q + (long)e_row[e] * p.q_st + (long)e_a[e] * p.q_sa;
    for (int r = lane; r < D; r += 64)
      Ql[e * QS + r] = ok ? qp[r] : (unsigned short)0;
  }

  const int e_s = tid >> 4, kk = tid & 15;    // softmax role
  const int my_pos = e_pos[e_s], my_lo = e_lo[e_s];
  const int nsplit = gridDim.y, split = blockIdx.y;
  float m_run = -INFINITY, l_run = 0.f;
  if (p.sinks != nullptr && my_pos >= 0 && split == 0) {
    m_run = p.sinks[e_a[e_s] / p.maps];
    l_run = 1.f;
  }
  const float slope = p.slopes != nullptr ? p.slopes[e_a[e_s] / p.maps] : 0.f;
  f32x4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int* bt = p.block_tables + (long)seq * p.maxb;
  const int last_page = jmax >> 4;
  const KeyWalk walk = key_walk(lo, jmax, p.keep_first, MKT);
  const int per = (walk.n + nsplit - 1) / nsplit;
  const int v_end = min(walk.n, (split + 1) * per);
  auto page_at = [&](int pg) {
    return (long)min(max(bt[min(pg, last_page)], 0), p.nblocks - 1);
  };
  // keys past jmax re-read key jmax (their weights are masked to zero below)
  auto key_row = [&](int k0, long blk) {
    const int key = min(k0 + wave * 16 + lc, jmax);
    return k_cache + ((blk * p.G + g) * BS + (key & 15)) * (long)p.KW + koff +
           lg * 8;
  };
  // 8 consecutive keys of one page; groups wholly past jmax read the last valid
  // page (weights there are zero)
  auto value_page = [&](int key, long blk) {
    return v_cache + (blk * p.G + g) * (long)VW * BS + (key & 15);
  };
  for (int v = split * per; v < v_end; ++v) {
    const int k0 = walk.tile(v) * MKT;
    __syncthreads();   // Ql staged / previous tile's Pl and als consumed
    {
      const unsigned short* qrow = Ql + lc * QS;
      f32x4 sacc{0.f, 0.f, 0.f, 0.f};
      const unsigned short* rowp = key_row(k0, page_at((k0 >> 4) + wave));
#pragma unroll 4
      for (int r = 0; r < D; r += 32) {
        const u16x8 a = *reinterpret_cast<const u16x8*>(qrow + r + lg * 8);
        const u16x8 b = *reinterpret_cast<const u16x8*>(rowp + r);
        sacc = ra_mfma(a, b, sacc);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Ss[(lg * 4 + r) * MSS + wave * 16 + lc] = sacc[r];
    }
    __syncthreads();
    {
      float sv[4];
      float mx = -INFINITY;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = k0 + kk + 16 * u;
        sv[u] = key_visible(j, my_pos, my_lo, p.keep_first)
                    ? scaled_score(Ss[e_s * MSS + kk + 16 * u], p) -
                          slope * (float)(my_pos - j)
                    : -INFINITY;
        mx = fmaxf(mx, sv[u]);
      }
#pragma unroll
      for (int m = 8; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, WAVE_SIZE));
      const float m_new = fmaxf(m_run, mx);
      float alpha = 1.f, psum = 0.f;
      if (m_new == -INFINITY) {
#pragma unroll
        for (int u = 0; u < 4; ++u) Pl[e_s * MPS + kk + 16 * u] = 0;
      } else {
        alpha = __expf(m_run - m_new);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float pv = __expf(sv[u] - m_new);
          Pl[e_s * MPS + kk + 16 * u] = f2bf(pv);
          psum += pv;
        }
      }
      psum = group16_reduce_sum(psum);
      l_run = l_run * alpha + psum;
      m_run = m_new;
      if (kk == 0) als[e_s] = alpha;
    }
    __syncthreads();
    {
      float ar[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) ar[r] = als[lg * 4 + r];
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][r] *= ar[r];
#pragma unroll
      for (int ks = 0; ks < MKT; ks += 32) {
        const u16x8 a =
            *reinterpret_cast<const u16x8*>(Pl + lc * MPS + ks + lg * 8);
        const int keyb = k0 + ks + lg * 8;
        const unsigned short* pt = value_page(keyb, page_at(keyb >> 4));
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const int ch = (wave + 4 * i) * 16 + lc;
          if ((wave + 4 * i) * 16 < VW) {       // uniform over the wave
            const u16x8 b = *reinterpret_cast<const u16x8*>(pt + (long)ch * BS);
            acc[i] = ra_mfma(a, b, acc[i]);
          }
        }
      }
    }
  }
  if (nsplit > 1) {
    const long slot = (long)blockIdx.x * nsplit + split;
    if (kk == 0) {
      ws_ml[(slot * G16 + e_s) * 2] = m_run;
      ws_ml[(slot * G16 + e_s) * 2 + 1] = l_run;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = lg * 4 + r;
      float* wp = ws_acc + (slot * G16 + e) * VW;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        const int ch = (wave + 4 * i) * 16 + lc;
        if (ch < VW) wp[ch] = acc[i][r];
      }
    }
    return;
  }
  if (kk == 0) lsum[e_s] = l_run;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int e = lg * 4 + r;
    if (e >= n_ent) continue;
    const float l = lsum[e];
    const float inv = (l > 0.f ? 1.0f / l : 0.f) *
                      head_gate_of<unsigned short>(p, e_row[e], e_a[e]);
    TO* op = out + (long)e_row[e] * p.o_st + (long)e_a[e] * p.o_sa;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      const int ch = (wave + 4 * i) * 16 + lc;
      if (ch < VW) stf(op + ch, acc[i][r] * inv);
    }
  }
}

// Heads of 128 channels on values of 80 to 128: every wave takes keys of its own, 32
// at a time, with a maximum and a sum of its own, and the four meet once, at the end,
// so that nothing waits at a barrier and a wave's next keys and these values (16 KB)
// are under way all the time. S^T = K Q^T in an order of the key rows (key_at) in which
// a lane's 8 weights of 32 keys are neighbours, as the value pages hold them: the
// weights stay in its registers. VT tiles of 16 channels, all of them loaded (ALL): behind
// a branch for each that VW may leave out, the wait for the keys takes in the values asked
// for behind them, and a step costs two latencies. Bound by memory, us, with the branches
// / without: 64 rows of 16 heads on 4 behind 200 to 3000 keys 54.5 / 51.4 (210 MB, cold), in
// a window of 1024 29.1 / 27.7 (118 MB; a workgroup to a tile of 64 keys, its scores and
// weights through the LDS with three barriers, took 34), 33 rows behind 1000 to 8000 in
// the window 26.1 / 23.6, 16 behind 300 to 1200 15.8 / 14.8, one behind 7000 20.8 /
// 19.2 (launch_mfma has where the branches stay). Eight waves for four, of half the keys
// each, are no faster (27.7, 11.6 for 12.0 behind 7000 in the window, 102 for 94).
template <typename TO, int VT, bool ALL>
__global__ __launch_bounds__(THREADS, 2) void paged_attn_waves_kernel(
    TO* __restrict__ out, const unsigned short* __restrict__ q,
    const unsigned short* __restrict__ k_cache,
    const unsigned short* __restrict__ v_cache, AttnArgs p,
    float* __restrict__ ws_acc, float* __restrict__ ws_ml) {
  constexpr int BS = 16, D = 128, DK = D / 32, WKT = 32, QS = D + 8;
  constexpr int OS = D + 4;                           // fp32 row of the sums
  __shared__ __attribute__((aligned(16))) unsigned short Ql[G16 * QS];
  __shared__ __attribute__((aligned(16))) float os[4][G16 * OS];
  __shared__ float ms[4][G16], ls[4][G16];
  __shared__ int e_pos[G16], e_lo[G16], e_row[G16], e_a[G16];

  int n_ent, seq, g, koff;
  if (!tile_setup(p, blockIdx.x, e_pos, e_lo, e_row, e_a, n_ent, seq, g, koff))
    return;
  __syncthreads();
  const int VW = p.VW;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, lg = lane >> 4;
  int jmax = -1, lo = 1 << 30;
#pragma unroll
  for (int e = 0; e < G16; ++e) {
    jmax = max(jmax, e_pos[e]);
    lo = min(lo, e_lo[e]);
  }
  jmax = __builtin_amdgcn_readfirstlane(jmax);
  lo = __builtin_amdgcn_readfirstlane(lo);
  for (int e = wave; e < G16; e += 4) {
    const bool ok = e < n_ent;
    const unsigned short* qp =
        q + (long)e_row[e] * p.q_st + (long)e_a[e] * p.q_sa;
    for (int r = lane; r < D; r += 64)
      Ql[e * QS + r] = ok ? qp[r] : (unsigned short)0;
  }
  __syncthreads();
  u16x8 qf[DK];
#pragma unroll
  for (int r = 0; r < DK; ++r)
    qf[r] = *reinterpret_cast<const u16x8*>(Ql + lc * QS + r * 32 + lg * 8);

  const int my_pos = e_pos[lc], my_lo = e_lo[lc];
  const int nsplit = gridDim.y, split = blockIdx.y;
  float m_run = -INFINITY, l_run = 0.f;               // l: of this lane's keys
  if (p.sinks != nullptr && my_pos >= 0 && split == 0 && wave == 0) {
    m_run = p.sinks[e_a[lc] / p.maps];
    l_run = lg == 0 ? 1.f : 0.f;
  }
  const float slope = p.slopes != nullptr ? p.slopes[e_a[lc] / p.maps] : 0.f;
  f32x4 acc[VT];                                      // channels 16 c + 4 lg .. of pair lc
#pragma unroll
  for (int c = 0; c < VT; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int* bt = p.block_tables + (long)seq * p.maxb;
  const int last_page = jmax >> 4;
  const KeyWalk walk = key_walk(lo, jmax, p.keep_first, WKT);
  const int part = split * 4 + wave, parts = nsplit * 4;
  const int v_begin = (int)((long)walk.n * part / parts);
  const int v_end = (int)((long)walk.n * (part + 1) / parts);
  auto page_at = [&](int pg) {
    return min(max(bt[min(pg, last_page)], 0), p.nblocks - 1);
  };
  // key of row lc of product t; keys past jmax re-read key jmax (their weights are 0)
  auto key_at = [&](int t) { return (lc >> 2) * 8 + t * 4 + (lc & 3); };
  u16x8 kreg[2][DK], vreg[VT];
  auto keys = [&](int k0, int pg0, int pg1) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int key = min(k0 + key_at(t), jmax);
      const long blk = lc >= 8 ? pg1 : pg0;
      const unsigned short* rowp =
          k_cache + ((blk * p.G + g) * BS + (key & 15)) * (long)p.KW + koff + lg * 8;
#pragma unroll
      for (int r = 0; r < DK; ++r)
        kreg[t][r] = *reinterpret_cast<const u16x8*>(rowp + r * 32);
    }
  };
  int pg0 = 0, pg1 = 0;                               // pages of the tile at hand
  if (v_begin < v_end) {
    const int k0 = walk.tile(v_begin) * WKT;
    pg0 = page_at(k0 >> 4);
    pg1 = page_at((k0 >> 4) + 1);
    keys(k0, pg0, pg1);
  }
  for (int v = v_begin; v < v_end; ++v) {
    const int k0 = walk.tile(v) * WKT;
    const int kn = walk.tile(min(v + 1, v_end - 1)) * WKT;
    const int nx0 = page_at(kn >> 4), nx1 = page_at((kn >> 4) + 1);
    {
      // 8 neighbouring keys of one page; those past jmax weigh nothing
      const long blk = lg >= 2 ? pg1 : pg0;
      const unsigned short* pt =
          v_cache + (blk * p.G + g) * (long)VW * BS + (lg & 1) * 8 + lc * BS;
#pragma unroll
      for (int c = 0; c < VT; ++c)           // ALL: the last ones once more behind VW
        if (ALL || c * 16 < VW)
          vreg[c] = *reinterpret_cast<const u16x8*>(
              pt + (ALL ? min(c * 16, VW - 16) : c * 16) * BS);
    }
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int r = 0; r < DK; ++r) s[t] = ra_mfma(kreg[t][r], qf[r], s[t]);
    }
    if (v + 1 < v_end) keys(kn, nx0, nx1);
    pg0 = nx0;
    pg1 = nx1;
    float sv[8], mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) sv[i] = s[i >> 2][i & 3] * p.scale;
    if (p.softcap > 0.f)
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[i] = p.softcap * tanhf(sv[i] / p.softcap);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int j = k0 + lg * 8 + i;
      sv[i] = key_visible(j, my_pos, my_lo, p.keep_first)
                  ? sv[i] - slope * (float)(my_pos - j)
                  : -INFINITY;
      mx = fmaxf(mx, sv[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE_SIZE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE_SIZE));
    const float m_new = fmaxf(m_run, mx);
    // before any key was seen from 0: those hidden weigh 0, a score that is no number
    // (the maximum leaves it out) shows
    const bool any = m_new != -INFINITY;
    const float m_ref = any ? m_new : 0.f;
    const float alpha = any ? __expf(m_run - m_ref) : 1.f;
    u16x8 w;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float pv = __expf(sv[i] - m_ref);
      w[i] = f2bf(pv);
      sum += pv;
    }
    l_run = l_run * alpha + sum;
    m_run = m_new;
    if (__any(alpha != 1.f)) {
#pragma unroll
      for (int c = 0; c < VT; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[c][r] *= alpha;
    }
#pragma unroll
    for (int c = 0; c < VT; ++c)
      if (ALL || c * 16 < VW) acc[c] = ra_mfma(vreg[c], w, acc[c]);
  }
  l_run += __shfl_xor(l_run, 16, WAVE_SIZE);
  l_run += __shfl_xor(l_run, 32, WAVE_SIZE);
  if (lg == 0) {
    ms[wave][lc] = m_run;
    ls[wave][lc] = l_run;
  }
  if (lc < n_ent) {
#pragma unroll
    for (int c = 0; c < VT; ++c)
      *reinterpret_cast<f32x4*>(&os[wave][lc * OS + c * 16 + lg * 4]) = acc[c];
  }
  __syncthreads();
  for (int i = tid; i < n_ent * (D / 4); i += THREADS) {
    const int e = i / (D / 4), ch = i % (D / 4) * 4;
    if (ch >= VW) continue;
    float M = -INFINITY;
#pragma unroll
    for (int u = 0; u < 4; ++u) M = fmaxf(M, ms[u][e]);
    const float ref = M == -INFINITY ? 0.f : M;
    float L = 0.f;
    f32x4 o{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 4; ++u) {            // without a maximum: 0, or no number
      const float f = __expf(ms[u][e] - ref);
      L += ls[u][e] * f;
      const f32x4 x = *reinterpret_cast<const f32x4*>(&os[u][e * OS + ch]);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] += x[r] * f;
    }
    if (nsplit > 1) {
      const long slot = (long)blockIdx.x * nsplit + split;
      if (ch == 0) {
        ws_ml[(slot * G16 + e) * 2] = M;
        ws_ml[(slot * G16 + e) * 2 + 1] = L;
      }
      *reinterpret_cast<f32x4*>(ws_acc + (slot * G16 + e) * VW + ch) = o;
    } else {
      const float inv = (L > 0.f ? 1.0f / L : 0.f) *
                        head_gate_of<unsigned short>(p, e_row[e], e_a[e]);
      TO* op = out + (long)e_row[e] * p.o_st + (long)e_a[e] * p.o_sa + ch;
#pragma unroll
      for (int r = 0; r < 4; ++r) stf(op + r, o[r] * inv);
    }
  }
}

// out = sum_s acc_s exp(m_s - M) / sum_s l_s exp(m_s - M) over a tile's
// splits; one workgroup of 128 lanes per (tile, pair)
constexpr int MERGE_THREADS = 128;

template <typename TO>
__global__ __launch_bounds__(MERGE_THREADS) void paged_attn_merge_kernel(
    TO* __restrict__ out, AttnArgs p, const float* __restrict__ ws_acc,
    const float* __restrict__ ws_ml, int nsplit) {
  const int* tl = p.tiles + (long)blockIdx.x * 6;
  const int row0 = tl[0], nrows = tl[1], a0 = tl[2], n_a = tl[3];
  const int seq = tl[4], a_step = tl[5];
  const int e = blockIdx.y;
  // the same test the attention kernel applies: skipped tiles left nothing
  if (row0 < 0 || nrows < 1 || row0 + nrows > p.T || a0 < 0 || n_a < 1 ||
      a_step < 1 || a0 + (long)(n_a - 1) * a_step >= p.A ||
      (long)nrows * n_a > G16 || seq < 0 || seq >= p.nseq ||
      (a0 / p.maps) / p.rep >= p.G || e >= nrows * n_a)
    return;
  const int VW = p.VW;
  const long base = (long)blockIdx.x * nsplit;
  float M = -INFINITY;
  for (int s = 0; s < nsplit; ++s)
    M = fmaxf(M, ws_ml[((base + s) * G16 + e) * 2]);
  // a part without a maximum saw no key and is 0, or has only scores that are no
  // numbers and is none itself
  const float ref = M == -INFINITY ? 0.f : M;
  float L = 0.f;
  for (int s = 0; s < nsplit; ++s) {
    const float* ml = ws_ml + ((base + s) * G16 + e) * 2;
    L += ml[1] * __expf(ml[0] - ref);
  }
  const int row = row0 + e / n_a, a = a0 + (e % n_a) * a_step;
  const float inv = (L > 0.f ? 1.0f / L : 0.f) *
                    head_gate_of<unsigned short>(p, row, a);
  TO* op = out + (long)row * p.o_st + (long)a * p.o_sa;
  for (int ch = threadIdx.x; ch < VW; ch += MERGE_THREADS) {
    float v = 0.f;
    for (int s = 0; s < nsplit; ++s)
      v += ws_acc[((base + s) * G16 + e) * VW + ch] *
           __expf(ws_ml[((base + s) * G16 + e) * 2] - ref);
    stf(op + ch, v * inv);
  }
}

// ---- prompts ---------------------------------------------------------------
// Portions of many rows, heads of 128 channels on values of 128, one map, pages
// of 16 keys: a workgroup takes 128 rows of one head, 4 waves x 32 rows, and
// walks the keys 64 at a time on v_mfma_f32_32x32x16_bf16, from the page pools.
//  - S^T = K Q^T: a lane holds scores of one row; keys are multiplied in an order
//    in which a lane's 8 of 16 are neighbours (key_of), so that the value pages,
//    channel by channel as they lie in the pool, are the operand of O^T = V^T P^T
//    with one 16-byte LDS read.
//  - pages go to the LDS by themselves, a wave brings one page of keys (16-byte
//    chunks XORed with the row) and one of values; two buffers of each, one
//    barrier a tile.
//  - a wave works on 32 keys at a time: the next 32 are multiplied while these
//    are weighted, so the K buffer of tile j holds keys 64 j + 32 .. 64 j + 95 and
//    the first 32 come before the loop. Pairs of whole tiles (no key of them
//    hidden from any row of the wave) run without masks.
//  - the running maximum is exact, as in the kernel above: the largest weight is
//    1 and rounds to itself. Let 2^8 above it, as prompts of the other models
//    do, the error of a row is 2.2e-3 instead of 1.5e-3 of its length.
// Bound by the latency of a tile's loads and its chain (1.9 us a tile of 64 keys
// where few workgroups run, 3.3 with two on every CU): 16 heads on 4, six prompts
// of 301 to 1900 rows in a window of 1024 with slopes 240 -> 85 us a layer, 8 x 200
// rows behind 2000 (32 heads on 8) 207 -> 64, 16 x 100 behind 100 37 -> 16.
typedef __attribute__((ext_vector_type(16))) float pr_f32x16;
typedef __attribute__((ext_vector_type(2))) unsigned int pr_u32x2;

constexpr int PR_ROWS = 128;       // rows of a workgroup
constexpr int PR_KEYS = 64;        // keys of a tile
constexpr int PR_D = 128;
constexpr float PR_LOG2E = 1.4426950408889634f;

struct PromptArgs {
  const int* block_tables;   // [nseq, maxb]
  const int* tiles;          // [5, ntiles] sequence's first row, tile's first
                             // row there, cached tokens, rows, sequence
  const float* sinks;        // [A] or null
  const float* slopes;       // [A] or null
  float scale;
  long q_st, o_st;           // row strides of q and out, heads packed
  int ntiles, T, A, G, nseq, maxb, nblocks, window;
};

__global__ __launch_bounds__(THREADS, 2) void paged_prompt_kernel(
    unsigned short* __restrict__ out, const unsigned short* __restrict__ q,
    const unsigned short* __restrict__ k_cache,
    const unsigned short* __restrict__ v_cache, PromptArgs p) {
  constexpr int D = PR_D, BS = 16, QK = D / 16, NT = D / 32, HB = 32;
  constexpr int TILE = PR_KEYS * D;        // elements of a buffer
  constexpr int PAGE = BS * D;
  __shared__ __attribute__((aligned(1024))) unsigned short lds[4 * TILE];

  // heads of one kv head on one XCD (workgroups go round the 8 XCDs)
  int a = blockIdx.x % p.A;
  if (p.A % 8 == 0) a = (a % 8) * (p.A / 8) + a / 8;
  const int tile = (gridDim.x - 1 - blockIdx.x) / p.A;
  const int row0 = p.tiles[tile], q0 = p.tiles[p.ntiles + tile];
  const int hist = p.tiles[2 * p.ntiles + tile];
  const int nnew = p.tiles[3 * p.ntiles + tile];
  const int seq = p.tiles[4 * p.ntiles + tile];
  if (row0 < 0 || hist < 0 || nnew < 1 || row0 + nnew > p.T || q0 < 0 ||
      q0 >= nnew || seq < 0 || seq >= p.nseq ||
      (hist + nnew + BS - 1) / BS > p.maxb)
    return;
  const int g = a / (p.A / p.G);
  const int len = hist + nnew;
  const int* bt = p.block_tables + (long)seq * p.maxb;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lc = lane & 31, hf = lane >> 5;
  const int qrow = q0 + wave * 32 + lc;            // within the new rows
  const int qpos = hist + qrow;
  u32x4 qf[QK];
  {
    const unsigned short* qp =
        q + (long)(row0 + min(qrow, nnew - 1)) * p.q_st + (long)a * D + hf * 8;
#pragma unroll
    for (int kk = 0; kk < QK; ++kk)
      qf[kk] = *reinterpret_cast<const u32x4*>(qp + kk * 16);
  }
  const float sc = p.scale * PR_LOG2E;
  const float slope = p.slopes != nullptr ? p.slopes[a] / p.scale : 0.f;
  float m = -INFINITY, l = 0.f;                    // m in powers of two
  pr_f32x16 o[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;

  const int lo_wave = hist + q0 + wave * 32;       // this wave's first row
  const bool idle = q0 + wave * 32 >= nnew;        // it has none
  const int kv_end = min(len, hist + q0 + PR_ROWS);
  const int nt = (kv_end + PR_KEYS - 1) / PR_KEYS;
  // first keys that any row of the workgroup, of the wave may see, and the
  // first that all rows of the wave see
  const int first = p.window > 0 ? max(0, hist + q0 - p.window + 1) : 0;
  const int first_wave = p.window > 0 ? max(0, lo_wave - p.window + 1) : 0;
  const int first_all = p.window > 0 ? max(0, lo_wave + 31 - p.window + 1) : 0;
  const int kt0 = first / PR_KEYS;
  // and what this lane's row sees
  const int seen_lo = p.window > 0 ? qpos - p.window + 1 : 0;
  const int seen_hi = min(qpos, len - 1);

  const int lr = lane >> 4, ch = lane & 15;
  const unsigned int koff = (unsigned)(lr * D + (ch ^ lr) * 8) * 2;
  auto page_of = [&](int key) {
    const int pg = min(key, len - 1) / BS;
    return ((long)min(max(bt[pg], 0), p.nblocks - 1) * p.G + g) * PAGE;
  };
  // a page behind the sequence's end is its last one again
  auto stage_keys = [&](int key0, unsigned short* to) {
    const int key = key0 + wave * BS;
    if (key < kt0 * PR_KEYS) return;
    const unsigned short* base = k_cache + page_of(key);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load_to_lds(base + i * 4 * D, koff ^ (i * 64), to + wave * PAGE + i * 4 * D);
  };
  auto stage_values = [&](int key0, unsigned short* to) {
    const unsigned short* base = v_cache + page_of(key0 + wave * BS);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      load_to_lds(base + i * 512, (unsigned)lane * 16, to + wave * PAGE + i * 512);
  };
  auto kbuf = [&](int j) { return lds + (j & 1) * TILE; };
  auto vbuf = [&](int j) { return lds + (2 + (j & 1)) * TILE; };

  // row lc of the K operand is key key_of(lc) of 32: a lane's scores r are keys
  // 16 (r>>3) + 8 hf + (r&7)
  const int key_of = (lc >> 4) * 16 + ((lc >> 2) & 1) * 8 + ((lc >> 3) & 1) * 4 +
                     (lc & 3);
  const unsigned short *ka[QK], *va = lds + 2 * TILE + lc * BS + hf * 8;
#pragma unroll
  for (int i = 0; i < QK; ++i)
    ka[i] = lds + key_of * D + (((i * 2 + hf) ^ (key_of & 15)) * 8);

  // unscaled scores of keys kv0 .. kv0 + 31, on top of slope * distance / scale;
  // at: elements from ka
  auto scores = [&](int at, int kv0, pr_f32x16& s) {
    const float near = slope * (float)(kv0 + 8 * hf - qpos);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      s[r] = __builtin_fmaf(slope, (float)(16 * (r >> 3) + (r & 7)), near);
#pragma unroll
    for (int kk = 0; kk < QK; ++kk)
      s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(ra_s16x8,
                             *reinterpret_cast<const u32x4*>(ka[kk] + at)),
          __builtin_bit_cast(ra_s16x8, qf[kk]), s, 0, 0, 0);
  };
  auto row_max = [&](const pr_f32x16& s) {          // in powers of two
    float x = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
    for (int r = 3; r < 15; r += 2) x = fmaxf(fmaxf(x, s[r]), s[r + 1]);
    x = fmaxf(x, s[15]);
    return half_wave_max(x) * sc;
  };
  auto rescale = [&](float mx) {
    if (__any(mx > m)) {
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
  auto weights = [&](const pr_f32x16& s, u32x4 (&pf)[2], float base) {
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float x = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[t * 8 + w * 2], sc, -base));
        const float y = __builtin_amdgcn_exp2f(
            __builtin_fmaf(s[t * 8 + w * 2 + 1], sc, -base));
        sum += x + y;
        const f32x2 xy{x, y};
        pf[t][w] = __builtin_bit_cast(unsigned int,
                                      __builtin_convertvector(xy, bf16x2));
      }
    l += sum;
  };
  // at: elements from va. CUT: only `left` keys of the 32 are the sequence's, and
  // what lies behind them in its last page is not multiplied.
  auto weigh = [&](int at, const u32x4 (&pf)[2], auto cut, int left) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        u32x4 v = *reinterpret_cast<const u32x4*>(va + at + t * PAGE + n * 512);
        if constexpr (decltype(cut)::value) {
          const int own = left - t * 16 - hf * 8;
#pragma unroll
          for (int w = 0; w < 4; ++w)
            v[w] &= own > 2 * w + 1 ? 0xffffffffu : own > 2 * w ? 0xffffu : 0u;
        }
        o[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
            __builtin_bit_cast(ra_s16x8, v),
            __builtin_bit_cast(ra_s16x8, pf[t]), o[n], 0, 0, 0);
      }
  };
  // Tile j is in the LDS for every wave, and every wave is done with tile
  // j - 1, whose buffers tile j + 1 takes.
  auto advance = [&](int j) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int next = (j + 1) * PR_KEYS;
    if (next + HB < kv_end) stage_keys(next + HB, kbuf(j + 1));
    if (next < kv_end) stage_values(next, vbuf(j + 1));
  };

  const int k0 = kt0 * PR_KEYS;
  stage_keys(k0 - HB, kbuf(kt0 + 1));
  if (k0 + HB < kv_end) stage_keys(k0 + HB, kbuf(kt0));
  stage_values(k0, vbuf(kt0));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  pr_f32x16 st;
  scores(((kt0 + 1) & 1) * TILE + HB * D, k0, st);

  float mx = 0.f;
  bool known = false;                              // mx is st's
  auto whole = [&](int j, int par) {               // par = j & 1, a constant
    advance(j);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float base = rescale(mx);
      pr_f32x16 next;
      u32x4 pf[2];
      scores(par * TILE + h * HB * D, j * PR_KEYS + (h + 1) * HB, next);
      weights(st, pf, base);
      weigh(par * TILE + h * 2 * PAGE, pf, std::false_type{}, 32);
      st = next;
      mx = row_max(st);
    }
  };
  // tiles whose every key every row of the wave sees, and their next tile exists
  const int whole_lo = (first_all + PR_KEYS - 1) / PR_KEYS;
  const int whole_hi = idle ? 0 : min(nt - 1, (lo_wave + 1) / PR_KEYS);
  for (int j = kt0; j < nt;) {
    if (!(j & 1) && j >= whole_lo && j + 1 < whole_hi) {
      if (!known) mx = row_max(st);
      known = true;
      whole(j, 0);
      whole(j + 1, 1);
      j += 2;
      continue;
    }
    known = false;
    advance(j);
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int kv0 = j * PR_KEYS + h * HB;
      if (kv0 > lo_wave + 31 || kv0 >= kv_end || idle) break;
      const int at = (j & 1) * TILE + h * HB * D;
      if (kv0 + HB > first_wave) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kv = kv0 + 16 * (r >> 3) + 8 * hf + (r & 7);
          st[r] = kv >= seen_lo && kv <= seen_hi ? st[r] : -INFINITY;
        }
        const float base = rescale(row_max(st));
        u32x4 pf[2];
        weights(st, pf, base);
        const int vat = (j & 1) * TILE + h * 2 * PAGE;
        if (len - kv0 < HB) weigh(vat, pf, std::true_type{}, len - kv0);
        else weigh(vat, pf, std::false_type{}, HB);
      }
      if (kv0 + HB < kv_end) scores(at, kv0 + HB, st);
    }
    ++j;
  }
  __syncthreads();

  l += __shfl_xor(l, 32, 64);
  float num = 1.f;
  if (p.sinks != nullptr) {                        // no key, no value
    const float sk = p.sinks[a] * PR_LOG2E;
    const float M = fmaxf(m, sk);
    num = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - M);
    l = l * num + __builtin_amdgcn_exp2f(sk - M);
  }
  const float inv = l > 0.f ? num / l : 0.f;
  // through the wave's own part of the LDS to whole rows
  unsigned short* ol = lds + wave * 32 * D;
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      pr_u32x2 w;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const f32x2 xy{o[n][rr * 4 + c * 2] * inv, o[n][rr * 4 + c * 2 + 1] * inv};
        w[c] = __builtin_bit_cast(unsigned int,
                                  __builtin_convertvector(xy, bf16x2));
      }
      *reinterpret_cast<pr_u32x2*>(
          ol + lc * D + ((n * 8 + rr * 2 + hf) ^ (lc & 15)) * 4) = w;
    }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    const int u = lane + i * 64, r = u / 16, c = u % 16;
    const pr_u32x2 x = *reinterpret_cast<const pr_u32x2*>(
        ol + r * D + ((2 * c) ^ (r & 15)) * 4);
    const pr_u32x2 y = *reinterpret_cast<const pr_u32x2*>(
        ol + r * D + ((2 * c + 1) ^ (r & 15)) * 4);
    const int row = q0 + wave * 32 + r;
    if (row < nnew)
      *reinterpret_cast<u32x4*>(out + (long)(row0 + row) * p.o_st + (long)a * D +
                                c * 8) = u32x4{x[0], x[1], y[0], y[1]};
  }
}

template <int NT, typename TO>
void launch_mfma(void* out, const void* q, const void* kc, const void* vc,
                 const AttnArgs& p, int ntiles, int nsplit, float* ws_acc,
                 float* ws_ml, hipStream_t s) {
  const size_t smem = (size_t)G16 * (p.D + 8) * 2 + (size_t)G16 * MPS * 2 +
                      (size_t)(G16 * MSS + 2 * G16) * sizeof(float);
  bool alone = false;
  if constexpr (NT == 2) {
    alone = p.D == 128;
    // About four tiles a CU of uneven lengths end with the longest, which the others'
    // values, all asked for at once, keep waiting; us, a branch for each / all: rows behind
    // 100 to 1500 keys in a window of 1024, 16 heads on 4, 800 tiles 65.8 / 64.3, 864 67.2
    // / 72.8, 1024 81.5 / 84.6, 1088 85.4 / 87.6, 1152 91.3 / 92.5, 1200 95.7 / 95.3 (but
    // 1024 behind 600 to 1200 95.4 / 91.6).
    const bool branch = ntiles > 816 && ntiles <= 1184;
#define WAVES(VT, ALL)                                                        \
  paged_attn_waves_kernel<TO, VT, ALL><<<dim3(ntiles, nsplit), THREADS, 0, s>>>( \
      (TO*)out, (const unsigned short*)q, (const unsigned short*)kc,          \
      (const unsigned short*)vc, p, ws_acc, ws_ml)
    if (alone && branch) WAVES(8, false);
    else if (alone && p.VW > 96) WAVES(8, true);
    else if (alone) WAVES(6, true);
#undef WAVES
  }
  if (!alone)
    paged_attn_mfma_kernel<NT, TO><<<dim3(ntiles, nsplit), THREADS, smem, s>>>(
        (TO*)out, (const unsigned short*)q, (const unsigned short*)kc,
        (const unsigned short*)vc, p, ws_acc, ws_ml);
  if (nsplit > 1)
    paged_attn_merge_kernel<TO><<<dim3(ntiles, G16), MERGE_THREADS, 0, s>>>(
        (TO*)out, p, ws_acc, ws_ml, nsplit);
}

template <typename TO>
void dispatch_mfma(void* out, const void* q, const void* kc, const void* vc,
                   const AttnArgs& p, int ntiles, int nsplit, float* ws_acc,
                   float* ws_ml, hipStream_t s) {
  const int nt = (p.VW / 16 + 3) / 4;
  if (nt <= 1) launch_mfma<1, TO>(out, q, kc, vc, p, ntiles, nsplit, ws_acc, ws_ml, s);
  else if (nt <= 2) launch_mfma<2, TO>(out, q, kc, vc, p, ntiles, nsplit, ws_acc, ws_ml, s);
  else if (nt <= 4) launch_mfma<4, TO>(out, q, kc, vc, p, ntiles, nsplit, ws_acc, ws_ml, s);
  else launch_mfma<8, TO>(out, q, kc, vc, p, ntiles, nsplit, ws_acc, ws_ml, s);
}

template <typename TQ, typename TC, typename TO, int NJ, int KT>
void launch_exact(void* out, const void* q, const void* kc, const void* vc,
                  const AttnArgs& p, int ntiles, hipStream_t s) {
  const size_t smem = (size_t)(G16 * p.D + KT * (p.D + 1) + KT * (p.VW + 1) +
                               G16 * KT + 2 * G16) * sizeof(float);
  auto kern = paged_attn_exact_kernel<TQ, TC, TO, NJ, KT>;
  if (smem > 48 * 1024)
    (void)hipFuncSetAttribute((const void*)kern,
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)smem);
  kern<<<ntiles, THREADS, smem, s>>>((TO*)out, (const TQ*)q, (const TC*)kc,
                                     (const TC*)vc, p);
}

template <typename TQ, typename TC, typename TO>
void dispatch_exact(void* out, const void* q, const void* kc, const void* vc,
                    const AttnArgs& p, int ntiles, hipStream_t s) {
  // wide heads take shorter key tiles so the staging fits the LDS
  const bool small = p.D + p.VW <= 320;   // KT = 32 within 64 KB
  if (p.VW <= 64) {
    if (small) launch_exact<TQ, TC, TO, 1, 32>(out, q, kc, vc, p, ntiles, s);
    else launch_exact<TQ, TC, TO, 1, 16>(out, q, kc, vc, p, ntiles, s);
  } else if (p.VW <= 128) {
    if (small) launch_exact<TQ, TC, TO, 2, 32>(out, q, kc, vc, p, ntiles, s);
    else launch_exact<TQ, TC, TO, 2, 16>(out, q, kc, vc, p, ntiles, s);
  } else if (p.VW <= 256) {
    if (small) launch_exact<TQ, TC, TO, 4, 32>(out, q, kc, vc, p, ntiles, s);
    else launch_exact<TQ, TC, TO, 4, 16>(out, q, kc, vc, p, ntiles, s);
  } else {
    launch_exact<TQ, TC, TO, 8, 16>(out, q, kc, vc, p, ntiles, s);
  }
}

}  // namespace

// largest head sizes the exact path's LDS tiling covers (the MFMA path
// takes score sizes up to 1024 and value sizes up to 512)
int paged_attn_max_dim() { return 512; }

// 1 when (q / pool dtype, page size, head sizes) take the MFMA path
int paged_attn_uses_mfma(int io_bf, int BS, int D, int VW) {
  return io_bf && BS == 16 && D % 32 == 0 && D <= 1024 && VW % 16 == 0 &&
         VW <= 512;
}

// q_bf: q and the pools are bf16, else fp32. out_bf: out is bf16, else fp32.
// nsplit > 1 (MFMA path only) needs ws_acc [ntiles*nsplit*16*VW] and ws_ml
// [ntiles*nsplit*16*2] fp32.
void paged_attention_launch(void* out, const void* q, const void* k_cache,
                            const void* v_cache, const int* block_tables,
                            const int* tiles, const int* pos32,
                            const float* sinks, const float* slopes,
                            float scale, float softcap, long q_st, long q_sa,
                            long o_st, long o_sa, int ntiles, int T,
                            int A, int D, int VW, int KW, int G, int BS,
                            int maps, int rep, int nseq, int maxb, int nblocks,
                            int window, int keep_first, int chunk,
                            const void* gate, long g_st, int q_bf, int out_bf,
                            int force_exact, int nsplit, float* ws_acc,
                            float* ws_ml, hipStream_t s) {
  if (ntiles == 0) return;
  AttnArgs p;
  p.block_tables = block_tables; p.tiles = tiles; p.pos32 = pos32;
  p.softcap = softcap; p.q_st = q_st; p.q_sa = q_sa; p.o_st = o_st;
  p.o_sa = o_sa;
  p.sinks = sinks; p.slopes = slopes; p.scale = scale; p.T = T; p.A = A; p.D = D; p.VW = VW;
  p.KW = KW; p.G = G; p.BS = BS; p.maps = maps; p.rep = rep; p.nseq = nseq;
  p.maxb = maxb; p.nblocks = nblocks; p.window = window;
  p.keep_first = keep_first; p.chunk = chunk; p.gate = gate; p.g_st = g_st;
  if (!force_exact && paged_attn_uses_mfma(q_bf, BS, D, VW)) {
    if (out_bf)
      dispatch_mfma<unsigned short>(out, q, k_cache, v_cache, p, ntiles, nsplit, ws_acc, ws_ml, s);
    else
      dispatch_mfma<float>(out, q, k_cache, v_cache, p, ntiles, nsplit, ws_acc, ws_ml, s);
    return;
  }
  if (q_bf) {
    if (out_bf)
      dispatch_exact<unsigned short, unsigned short, unsigned short>(out, q, k_cache, v_cache, p, ntiles, s);
    else
      dispatch_exact<unsigned short, unsigned short, float>(out, q, k_cache, v_cache, p, ntiles, s);
  } else {
    dispatch_exact<float, float, float>(out, q, k_cache, v_cache, p, ntiles, s);
  }
}

void paged_prompt_attention_launch(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const int* block_tables, const int* tiles, const float* sinks,
    const float* slopes, float scale, long q_st, long o_st, int ntiles, int T,
    int A, int G, int nseq, int maxb, int nblocks, int window, hipStream_t s) {
  if (ntiles == 0) return;
  PromptArgs p;
  p.block_tables = block_tables; p.tiles = tiles; p.sinks = sinks;
  p.slopes = slopes; p.scale = scale; p.q_st = q_st; p.o_st = o_st;
  p.ntiles = ntiles; p.T = T; p.A = A; p.G = G; p.nseq = nseq; p.maxb = maxb;
  p.nblocks = nblocks; p.window = window;
  paged_prompt_kernel<<<dim3((unsigned)ntiles * A), THREADS, 0, s>>>(
      (unsigned short*)out, (const unsigned short*)q,
      (const unsigned short*)k_cache, (const unsigned short*)v_cache, p);
}
