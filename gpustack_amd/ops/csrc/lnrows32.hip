// Row kernels of the pre-norm fp32 stream with layer norms, of attention
// without rotation, and of scored expert routing (gfx950).
//
// The stream x [T, W] is fp32 and updated in place; statistics, norms, the
// query temperature and router scores are fp32 whatever the GEMM dtype is,
// and every kernel emits its GEMM operand in that dtype directly.
//
//   embed_rows_scaled : x = embed[token] * scale
//   add_layer_norm    : x += a;  h = (x - mean) / sqrt(var + eps) * w + b
//                       (closes one sublayer and opens the next in one
//                       pass; the row stays in registers between the two)
//   head_norm_store   : weighted RMS norm of every q / k head, query
//                       temperature, value blend, q out, k (and v) into
//                       their paged pools
//   route_topk        : sigmoid / softmax scores, choice correction,
//                       groups ranked by their best few, top-k, weights
#include "common.h"

namespace {

template <typename T> DEVICE_INLINE float ld(const T* p);
template <> DEVICE_INLINE float ld<float>(const float* p) { return *p; }
template <> DEVICE_INLINE float ld<unsigned short>(const unsigned short* p) {
  return bf2f(*p);
}
template <typename T> DEVICE_INLINE void st(T* p, float v);
template <> DEVICE_INLINE void st<float>(float* p, float v) { *p = v; }
template <> DEVICE_INLINE void st<unsigned short>(unsigned short* p, float v) {
  *p = f2bf(v);
}

constexpr int ROW_THREADS = 256;

DEVICE_INLINE float block_sum(float v, float* red) {
  v = wave_reduce_sum(v);
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

template <typename TW>
__global__ __launch_bounds__(ROW_THREADS) void embed_rows_scaled_kernel(
    float* __restrict__ x, const long* __restrict__ tokens,
    const TW* __restrict__ embed, int W, long vocab, float scale) {
  const long t = blockIdx.x;
  const long tok = min(max(tokens[t], 0L), vocab - 1);   // never read outside
  const TW* e = embed + tok * W;
  for (int i = threadIdx.x; i < W; i += ROW_THREADS)
    x[t * W + i] = ld(e + i) * scale;
}

// The same for bf16 rows of a multiple of 8 at 16-byte addresses: 7032 rows of 2048
// 19.8 us (a value a lane and step 31).
__global__ __launch_bounds__(ROW_THREADS) void embed_rows_vec_kernel(
    float* __restrict__ x, const long* __restrict__ tokens,
    const unsigned short* __restrict__ embed, int W, long vocab, float scale) {
  const long t = blockIdx.x;
  const long tok = min(max(tokens[t], 0L), vocab - 1);   // never read outside
  const unsigned short* e = embed + tok * W;
  for (int i = threadIdx.x * 8; i < W; i += ROW_THREADS * 8) {
    float f[8];
    bf8_to_f32(*reinterpret_cast<const u16x8*>(e + i), f);
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] *= scale;
    f32x4* to = reinterpret_cast<f32x4*>(x + t * W + i);
    to[0] = f32x4{f[0], f[1], f[2], f[3]};
    to[1] = f32x4{f[4], f[5], f[6], f[7]};
  }
}

// NV: row values each lane keeps in registers (W <= NV * 256); wider rows
// re-read x. Mean first, then the mean of the squared deviations.
template <typename TA, typename TH, int NV>
__global__ __launch_bounds__(ROW_THREADS) void add_layer_norm_kernel(
    float* __restrict__ x, const TA* __restrict__ a,
    const float* __restrict__ w, const float* __restrict__ b,
    TH* __restrict__ h, int W, float eps) {
  __shared__ float red[4];
  const long t = blockIdx.x;
  float* xr = x + t * W;
  float keep[NV];
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = threadIdx.x + j * ROW_THREADS;
    float v = 0.f;
    if (i < W) {
      v = xr[i];
      if (a != nullptr) {
        v += ld(a + t * W + i);
        xr[i] = v;
      }
    }
    keep[j] = v;
    sum += v;
  }
  for (int i = threadIdx.x + NV * ROW_THREADS; i < W; i += ROW_THREADS) {
    float v = xr[i];
    if (a != nullptr) {
      v += ld(a + t * W + i);
      xr[i] = v;
    }
    sum += v;
  }
  if (w == nullptr) return;
  const float mean = block_sum(sum, red) / (float)W;
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = threadIdx.x + j * ROW_THREADS;
    if (i < W) {
      const float d = keep[j] - mean;
      sq += d * d;
    }
  }
  for (int i = threadIdx.x + NV * ROW_THREADS; i < W; i += ROW_THREADS) {
    const float d = xr[i] - mean;
    sq += d * d;
  }
  const float inv = 1.0f / sqrtf(block_sum(sq, red) / (float)W + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = threadIdx.x + j * ROW_THREADS;
    if (i < W) st(h + t * W + i, (keep[j] - mean) * inv * w[i] + b[i]);
  }
  for (int i = threadIdx.x + NV * ROW_THREADS; i < W; i += ROW_THREADS)
    st(h + t * W + i, (xr[i] - mean) * inv * w[i] + b[i]);
}

// The same for rows of a multiple of 8 at 16-byte addresses, up to 8192: a lane
// holds 8 NV neighbours, 16 bytes a load. FROM says what is added: nothing, bf16
// or fp32 rows, or the fp32 parts [parts, T, W] of a product cut over k, rounded
// to bf16 as its join would (4.7 us a launch).
// Bound by the row's bytes, few rows by the launch: 7032 rows of 2048 45 -> 32 us
// (5.4 TB/s), 64 rows 7.4 -> 4.9, in four parts 4.7 + 7.4 -> 5.0.
// pick (or null): h's row t is the norm of row pick[t] of the N, and the sum goes
// nowhere: the stream's end, of the rows whose logits are asked for. One launch
// for the last sum, the gather and the norm: 64 rows of 2048 4.7 + 4.7 + 4.7 -> 5.
// Picks out of range, which the caller refuses (ForwardMeta.checked), are clamped.
enum AddFrom { NOTHING, ROWS16, ROWS32, PARTS };

template <typename TH, int NV, int FROM>
__global__ __launch_bounds__(ROW_THREADS) void add_layer_norm_vec_kernel(
    float* __restrict__ x, const void* __restrict__ a, int parts,
    const float* __restrict__ w, const float* __restrict__ b,
    TH* __restrict__ h, const long* __restrict__ pick, int N, int W, float eps) {
  __shared__ float red[4];
  long t = blockIdx.x;
  if (pick != nullptr) {
    t = pick[blockIdx.x];
    if (t < 0) t += N;
    t = t < 0 ? 0 : t < N ? t : N - 1;
  }
  float* xr = x + t * W;
  float keep[NV][8];
  // the weights come with the row and not behind its sums
  f32x4 wk[NV][2], bk[NV][2];
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (threadIdx.x + j * ROW_THREADS) * 8;
#pragma unroll
    for (int k = 0; k < 8; ++k) keep[j][k] = 0.f;
    if (i >= W) continue;
    if (w != nullptr) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        wk[j][k / 4][k % 4] = w[i + k];
        bk[j][k / 4][k % 4] = b[i + k];
      }
    }
    const f32x4 lo = *reinterpret_cast<const f32x4*>(xr + i);
    const f32x4 hi = *reinterpret_cast<const f32x4*>(xr + i + 4);
    float f[8];
    if constexpr (FROM == ROWS16) {
      bf8_to_f32(*reinterpret_cast<const u16x8*>(
                     (const unsigned short*)a + t * W + i), f);
    } else if constexpr (FROM == ROWS32) {
#pragma unroll
      for (int k = 0; k < 8; ++k) f[k] = ((const float*)a)[t * W + i + k];
    } else if constexpr (FROM == PARTS) {
      bf8_to_f32(join_parts8((const float*)a + t * W + i, (long)N * W, parts), f);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      float v = k < 4 ? lo[k] : hi[k - 4];
      if constexpr (FROM != NOTHING) v += f[k];
      keep[j][k] = v;
      sum += v;
    }
    if (FROM != NOTHING && pick == nullptr) {
      *reinterpret_cast<f32x4*>(xr + i) =
          f32x4{keep[j][0], keep[j][1], keep[j][2], keep[j][3]};
      *reinterpret_cast<f32x4*>(xr + i + 4) =
          f32x4{keep[j][4], keep[j][5], keep[j][6], keep[j][7]};
    }
  }
  if (w == nullptr) return;
  TH* hr = h + (long)blockIdx.x * W;
  const float mean = block_sum(sum, red) / (float)W;
  float sq = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
    if ((threadIdx.x + j * ROW_THREADS) * 8 < W)
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float d = keep[j][k] - mean;
        sq += d * d;
      }
  const float inv = 1.0f / sqrtf(block_sum(sq, red) / (float)W + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (threadIdx.x + j * ROW_THREADS) * 8;
    if (i >= W) continue;
    float f[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) 
      f[k] = (keep[j][k] - mean) * inv * wk[j][k / 4][k % 4] + bk[j][k / 4][k % 4];
    if constexpr (sizeof(TH) == 2) {
      *reinterpret_cast<u16x8*>(hr + i) = f32_to_bf8(f);
    } else {
      *reinterpret_cast<f32x4*>(hr + i) = f32x4{f[0], f[1], f[2], f[3]};
      *reinterpret_cast<f32x4*>(hr + i + 4) = f32x4{f[4], f[5], f[6], f[7]};
    }
  }
}

// One workgroup per row; a wave takes one head at a time. Heads 0..HQ-1 are
// the queries, HQ..HQ+G-1 the keys; then the values, channel by channel.
// flags bit 0: values are stored by a later page-wise pass (the blend, if
// any, is written back into qkv for it).
template <typename TS, typename TC>
__global__ __launch_bounds__(ROW_THREADS) void head_norm_store_kernel(
    TS* __restrict__ q_out, TS* __restrict__ qkv, long ld_qkv, int nq, int nk,
    int nv, const float* __restrict__ q_w, const float* __restrict__ k_w,
    int D, float temp_coef, float temp_every, const int* __restrict__ pos32,
    const TS* __restrict__ v_first, long ld_vf, const float* __restrict__ lam,
    TC* __restrict__ k_cache, TC* __restrict__ v_cache,
    const long* __restrict__ slots, long nslots, int G, int BS, int VW,
    float eps, int flags) {
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  TS* row = qkv + t * ld_qkv;
  const long slot = slots[t];
  const bool keep = slot >= 0 && slot < nslots;
  const long blk = keep ? slot / BS : 0;
  const int off = keep ? (int)(slot % BS) : 0;
  float temp = 1.f;
  if (temp_every > 0.f) {
    // exact for whole-numbered steps while the position is below 2^24
    const int p = max(pos32[t], 0);
    temp = 1.f + temp_coef * logf(floorf((float)(p + 1) / temp_every) + 1.f);
  }
  const int HQ = nq / D;
  for (int hd = wave; hd < HQ + G; hd += 4) {
    const bool is_q = hd < HQ;
    const TS* src = row + (long)hd * D;      // q heads then k heads, in order
    float ss = 0.f;
    for (int c = lane; c < D; c += 64) {
      const float v = ld(src + c);
      ss += v * v;
    }
    ss = wave_reduce_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
    if (is_q) {
      TS* dst = q_out + t * nq + (long)hd * D;
      for (int c = lane; c < D; c += 64)
        st(dst + c, ld(src + c) * inv * q_w[c] * temp);
    } else if (keep) {
      TC* dst = k_cache + ((blk * G + (hd - HQ)) * BS + off) * (long)D;
      for (int c = lane; c < D; c += 64) st(dst + c, ld(src + c) * inv * k_w[c]);
    }
  }
  const bool later = flags & 1;
  if (later && v_first == nullptr) return;
  const float l = v_first != nullptr ? lam[0] : 0.f;
  TS* vr = row + nq + nk;
  for (int c = threadIdx.x; c < nv; c += ROW_THREADS) {
    float v = ld(vr + c);
    if (v_first != nullptr)
      v = (1.f - l) * v + l * ld(v_first + t * ld_vf + c);
    if (later) {
      st(vr + c, v);
    } else if (keep) {
      st(v_cache + ((blk * G + c / VW) * (long)VW + c % VW) * BS + off, v);
    }
  }
}

// The same for bf16 rows at 16-byte addresses with heads of 64, 128 or 256
// channels: LPH lanes share a head, 8 channels each, and 256 / LPH heads of any
// rows a workgroup. What a lane brings it reads once. Bound by the row's bytes,
// few rows by the launch: 64 rows of 16 + 2 x 4 heads of 128 11.6 -> 5.2 us,
// 7032 rows 48 -> 25 (a wave a head at a time, 2 bytes a lane, two passes).
// PARTS: the rows are fp32 parts of the projection, `stride` apart, added up in their
// order and rounded as the product's own join does it; the values are left in qkv.
template <int LPH, bool PARTS>
__global__ __launch_bounds__(ROW_THREADS) void head_norm_store_vec_kernel(
    unsigned short* __restrict__ q_out, unsigned short* __restrict__ qkv,
    const float* __restrict__ parts, long stride, int nparts, long ld_qkv, int nq, int nk, int nv, const float* __restrict__ q_w,
    const float* __restrict__ k_w, float temp_coef, float temp_every,
    const int* __restrict__ pos32, const unsigned short* __restrict__ v_first,
    long ld_vf, const float* __restrict__ lam,
    unsigned short* __restrict__ k_cache, unsigned short* __restrict__ v_cache,
    const long* __restrict__ slots, long nslots, int G, int BS, int VW,
    float eps, int flags, long units, int H) {
  constexpr int D = LPH * 8;
  const long u = (long)blockIdx.x * (ROW_THREADS / LPH) + threadIdx.x / LPH;
  if (u >= units) return;                      // whole heads leave together
  const long t = u / H;
  const int h = (int)(u % H), c = threadIdx.x % LPH * 8;
  const int HQ = nq / D;
  unsigned short* row = qkv + t * ld_qkv;
  const long slot = slots[t];
  const bool keep = slot >= 0 && slot < nslots;
  const long blk = keep ? slot / BS : 0;
  const int off = keep ? (int)(slot % BS) : 0;
  float f[8];
  auto mine = [&](int col) {
    if constexpr (PARTS)
      return join_parts8(parts + t * (nq + nk + nv) + col, stride, nparts);
    else
      return *reinterpret_cast<const u16x8*>(row + col);
  };
  if (h < HQ + G) {
    bf8_to_f32(mine(h * D + c), f);
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) ss += f[k] * f[k];
#pragma unroll
    for (int m = LPH / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, WAVE_SIZE);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
    const float* w = (h < HQ ? q_w : k_w) + c;
    float temp = 1.f;
    if (h < HQ && temp_every > 0.f) {
      // exact for whole-numbered steps while the position is below 2^24
      const int p = max(pos32[t], 0);
      temp = 1.f + temp_coef * logf(floorf((float)(p + 1) / temp_every) + 1.f);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      f[k] = f[k] * inv * w[k];
      if (h < HQ) f[k] *= temp;
    }
    if (h < HQ)
      *reinterpret_cast<u16x8*>(q_out + t * nq + (long)h * D + c) = f32_to_bf8(f);
    else if (keep)
      *reinterpret_cast<u16x8*>(
          k_cache + ((blk * G + (h - HQ)) * BS + off) * (long)D + c) =
          f32_to_bf8(f);
    return;
  }
  const int vc = (h - HQ - G) * D + c;
  const bool later = flags & 1;
  if (vc >= nv || (!PARTS && later && v_first == nullptr)) return;
  unsigned short* vr = row + nq + nk + vc;
  u16x8 v = mine(nq + nk + vc);
  if (v_first != nullptr) {
    const float l = lam[0];
    float g[8];
    bf8_to_f32(v, f);
    bf8_to_f32(*reinterpret_cast<const u16x8*>(v_first + t * ld_vf + vc), g);
#pragma unroll
    for (int k = 0; k < 8; ++k) f[k] = (1.f - l) * f[k] + l * g[k];
    v = f32_to_bf8(f);
  }
  if (later || PARTS) *reinterpret_cast<u16x8*>(vr) = v;
  if (!later && keep) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v_cache[((blk * G + (vc + k) / VW) * (long)VW + (vc + k) % VW) * BS + off] =
          v[k];
  }
}

// (value, index) argmax over a wave; ties go to the lower index
DEVICE_INLINE void wave_argmax(float& v, int& idx) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) {
    const float ov = __shfl_xor(v, m, WAVE_SIZE);
    const int oi = __shfl_xor(idx, m, WAVE_SIZE);
    if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
  }
}

constexpr int NONE = 0x7fffffff;

// One wave per token. smem: score[E], choice[E], gscore[G], then flags
// taken[E] and gkept[G] (ints). Choice scores may be negative, so taken
// experts and groups carry flags instead of marker values.
__global__ __launch_bounds__(64) void route_topk_kernel(
    int* __restrict__ experts, float* __restrict__ weights,
    const float* __restrict__ logits, int ld_logits,
    const float* __restrict__ correction, int E, int G, int keep,
    int group_top, int top, int use_sigmoid, int renorm, float scale) {
  extern __shared__ float sm[];
  float* score = sm;
  float* choice = score + E;
  float* gscore = choice + E;
  int* taken = reinterpret_cast<int*>(gscore + G);
  int* gkept = taken + E;
  const long t = blockIdx.x;
  const int lane = threadIdx.x;
  const float* z = logits + t * ld_logits;
  if (use_sigmoid) {
    for (int e = lane; e < E; e += 64) score[e] = 1.0f / (1.0f + expf(-z[e]));
  } else {
    float mx = -INFINITY;
    for (int e = lane; e < E; e += 64) mx = fmaxf(mx, z[e]);
    mx = wave_reduce_max(mx);
    float sum = 0.f;
    for (int e = lane; e < E; e += 64) {
      const float p = expf(z[e] - mx);
      score[e] = p;
      sum += p;
    }
    sum = wave_reduce_sum(sum);
    const float inv = 1.0f / sum;
    for (int e = lane; e < E; e += 64) score[e] *= inv;
  }
  for (int e = lane; e < E; e += 64) {
    choice[e] = score[e] + (correction != nullptr ? correction[e] : 0.f);
    taken[e] = 0;
  }
  __syncthreads();
  const int per = E / G;
  if (G > 1 && keep < G) {
    for (int g = lane; g < G; g += 64) {
      // sum of the group's group_top largest choice scores: repeated
      // selection with a "used below this rank" bound on (value, index)
      float total = 0.f;
      float pv = INFINITY;
      int pi = -1;
      const int n = min(group_top, per);
      for (int it = 0; it < n; ++it) {
        float bv = -INFINITY;
        int bi = NONE;
        for (int j = 0; j < per; ++j) {
          const float c = choice[g * per + j];
          const bool after = c < pv || (c == pv && j > pi);
          if (after && (c > bv || (c == bv && j < bi) || bi == NONE)) {
            bv = c;
            bi = j;
          }
        }
        if (bi == NONE) break;
        total += bv;
        pv = bv;
        pi = bi;
      }
      gscore[g] = total;
      gkept[g] = 0;
    }
    __syncthreads();
    for (int it = 0; it < keep; ++it) {
      float v = -INFINITY;
      int gi = NONE;
      for (int g = lane; g < G; g += 64)
        if (!gkept[g] && (gi == NONE || gscore[g] > v)) { v = gscore[g]; gi = g; }
      wave_argmax(v, gi);
      // lanes without a candidate carry (-inf, NONE); a real candidate of
      // value -inf still wins by its lower index
      if (lane == 0 && gi != NONE) gkept[gi] = 1;
      __syncthreads();
    }
  } else {
    for (int g = lane; g < G; g += 64) gkept[g] = 1;
    __syncthreads();
  }
  float wsum = 0.f;
  for (int it = 0; it < top; ++it) {
    float v = -INFINITY;
    int ei = NONE;
    for (int e = lane; e < E; e += 64)
      if (!taken[e] && gkept[e / per] && (ei == NONE || choice[e] > v)) {
        v = choice[e];
        ei = e;
      }
    wave_argmax(v, ei);
    const bool ok = ei != NONE;       // host checks keep * per >= top
    const float s = ok ? score[ei] : 0.f;
    wsum += s;
    if (lane == 0) {
      experts[t * top + it] = ok ? ei : 0;
      weights[t * top + it] = s;
      if (ok) taken[ei] = 1;
    }
    __syncthreads();
  }
  const float mul = renorm ? scale / (wsum + 1e-20f) : scale;
  for (int it = lane; it < top; it += 64) weights[t * top + it] *= mul;
}

template <typename TA, typename TH>
void aln_pick(float* x, const void* a, const float* w, const float* b, void* h,
              int T, int W, float eps, hipStream_t s) {
  if (W <= 1024)
    add_layer_norm_kernel<TA, TH, 4><<<T, ROW_THREADS, 0, s>>>(
        x, (const TA*)a, w, b, (TH*)h, W, eps);
  else if (W <= 2048)
    add_layer_norm_kernel<TA, TH, 8><<<T, ROW_THREADS, 0, s>>>(
        x, (const TA*)a, w, b, (TH*)h, W, eps);
  else
    add_layer_norm_kernel<TA, TH, 16><<<T, ROW_THREADS, 0, s>>>(
        x, (const TA*)a, w, b, (TH*)h, W, eps);
}

template <typename TH, int NV>
void aln_vec(float* x, const void* a, int from, int parts, const float* w,
             const float* b, void* h, const long* pick, int T, int N, int W,
             float eps, hipStream_t s) {
#define ALN(F)                                                               \
  add_layer_norm_vec_kernel<TH, NV, F><<<T, ROW_THREADS, 0, s>>>(            \
      x, a, parts, w, b, (TH*)h, pick, N, W, eps)
  if (from == NOTHING) ALN(NOTHING);
  else if (from == ROWS16) ALN(ROWS16);
  else if (from == ROWS32) ALN(ROWS32);
  else ALN(PARTS);
#undef ALN
}

template <typename TH>
void aln_vec_pick(float* x, const void* a, int from, int parts, const float* w,
                  const float* b, void* h, const long* pick, int T, int N,
                  int W, float eps, hipStream_t s) {
#define ALN_ARGS x, a, from, parts, w, b, h, pick, T, N, W, eps, s
  if (W <= 2048) aln_vec<TH, 1>(ALN_ARGS);
  else if (W <= 4096) aln_vec<TH, 2>(ALN_ARGS);
  else aln_vec<TH, 4>(ALN_ARGS);
#undef ALN_ARGS
}

}  // namespace

// ---- launchers: `bf` flags say which operands are bf16 (else fp32) ----------

void embed_rows_scaled_launch(float* x, const long* tokens, const void* embed,
                              int T, int W, long vocab, float scale, int bf,
                              hipStream_t s) {
  if (T <= 0) return;
  if (bf && W % 8 == 0 && ((uintptr_t)x | (uintptr_t)embed) % 16 == 0)
    embed_rows_vec_kernel<<<T, ROW_THREADS, 0, s>>>(
        x, tokens, (const unsigned short*)embed, W, vocab, scale);
  else if (bf)
    embed_rows_scaled_kernel<unsigned short><<<T, ROW_THREADS, 0, s>>>(
        x, tokens, (const unsigned short*)embed, W, vocab, scale);
  else
    embed_rows_scaled_kernel<float><<<T, ROW_THREADS, 0, s>>>(
        x, tokens, (const float*)embed, W, vocab, scale);
}

// parts: of a [parts, N, W] in fp32, or 0 for rows [N, W]. pick: null (T = N),
// or the T rows whose norm h gets, x being left as it is. Returns 0 when parts or
// picked rows come with rows that only the general form takes.
int add_layer_norm_launch(float* x, const void* a, int parts, const float* w,
                          const float* b, void* h, const long* pick, int T,
                          int N, int W, float eps, int a_bf, int h_bf,
                          hipStream_t s) {
  if (T <= 0) return 1;
  const uintptr_t at = (uintptr_t)x | (uintptr_t)a | (uintptr_t)w |
                       (uintptr_t)b | (uintptr_t)h;
  if (W % 8 == 0 && W <= 8192 && at % 16 == 0) {
    const int from = a == nullptr ? NOTHING : parts > 0 ? PARTS
                   : a_bf ? ROWS16 : ROWS32;
    if (h_bf) aln_vec_pick<unsigned short>(x, a, from, parts, w, b, h, pick, T, N, W, eps, s);
    else aln_vec_pick<float>(x, a, from, parts, w, b, h, pick, T, N, W, eps, s);
    return 1;
  }
  if (parts > 0 || pick != nullptr) return 0;
  if (a_bf) {
    if (h_bf) aln_pick<unsigned short, unsigned short>(x, a, w, b, h, T, W, eps, s);
    else aln_pick<unsigned short, float>(x, a, w, b, h, T, W, eps, s);
  } else {
    if (h_bf) aln_pick<float, unsigned short>(x, a, w, b, h, T, W, eps, s);
    else aln_pick<float, float>(x, a, w, b, h, T, W, eps, s);
  }
  return 1;
}

// parts: the rows [T, nq + nk + nv] as fp32 parts [nparts, T, ..], or null. Returns 0
// where they are given and the kernel of whole lanes does not take the call.
int head_norm_store_launch(void* q_out, void* qkv, const float* parts, int nparts,
                           long ld_qkv, int nq, int nk, int nv, const float* q_w,
                           const float* k_w, int D, float temp_coef,
                           float temp_every, const int* pos32,
                           const void* v_first, long ld_vf, const float* lam,
                           void* k_cache, void* v_cache, const long* slots,
                           long nslots, int G, int BS, int VW, float eps,
                           int flags, int T, int bf, hipStream_t s) {
  if (T <= 0) return 1;
  const uintptr_t at = (uintptr_t)q_out | (uintptr_t)qkv | (uintptr_t)v_first |
                       (uintptr_t)k_cache | (uintptr_t)parts |
                       (uintptr_t)(ld_qkv * 2) |
                       (uintptr_t)(v_first != nullptr ? ld_vf * 2 : 0);
  if (bf && (D == 64 || D == 128 || D == 256) && nq % D == 0 && nk == G * D &&
      nv % 8 == 0 && at % 16 == 0) {
    const int H = nq / D + G + (nv + D - 1) / D;
    const long units = (long)T * H;
    const int per = ROW_THREADS / (D / 8);
    const dim3 grid((unsigned)((units + per - 1) / per));
#define HNS(L, P)                                                            \
  head_norm_store_vec_kernel<L, P><<<grid, ROW_THREADS, 0, s>>>(             \
      (unsigned short*)q_out, (unsigned short*)qkv, parts,                   \
      (long)T * (nq + nk + nv), nparts, ld_qkv, nq, nk, nv, q_w, k_w,        \
      temp_coef, temp_every, pos32, (const unsigned short*)v_first, ld_vf,   \
      lam, (unsigned short*)k_cache, (unsigned short*)v_cache, slots,        \
      nslots, G, BS, VW, eps, flags, units, H)
#define HNS_D(P)                                                             \
  if (D == 64) HNS(8, P);                                                    \
  else if (D == 128) HNS(16, P);                                             \
  else HNS(32, P)
    if (parts != nullptr) {
      HNS_D(true);
    } else {
      HNS_D(false);
    }
#undef HNS_D
#undef HNS
    return 1;
  }
  if (parts != nullptr) return 0;
  if (bf)
    head_norm_store_kernel<unsigned short, unsigned short>
        <<<T, ROW_THREADS, 0, s>>>(
            (unsigned short*)q_out, (unsigned short*)qkv, ld_qkv, nq, nk, nv,
            q_w, k_w, D, temp_coef, temp_every, pos32,
            (const unsigned short*)v_first, ld_vf, lam,
            (unsigned short*)k_cache, (unsigned short*)v_cache, slots, nslots,
            G, BS, VW, eps, flags);
  else
    head_norm_store_kernel<float, float><<<T, ROW_THREADS, 0, s>>>(
        (float*)q_out, (float*)qkv, ld_qkv, nq, nk, nv, q_w, k_w, D, temp_coef,
        temp_every, pos32, (const float*)v_first, ld_vf, lam, (float*)k_cache,
        (float*)v_cache, slots, nslots, G, BS, VW, eps, flags);
  return 1;
}

void route_topk_launch(int* experts, float* weights, const float* logits,
                       int ld_logits, const float* correction, int T, int E,
                       int G, int keep, int group_top, int top, int use_sigmoid,
                       int renorm, float scale, hipStream_t s) {
  if (T <= 0) return;
  const size_t smem = (size_t)(3 * E + 2 * G) * sizeof(float);
  route_topk_kernel<<<T, 64, smem, s>>>(experts, weights, logits, ld_logits,
                                        correction, E, G, keep, group_top, top,
                                        use_sigmoid, renorm, scale);
}
