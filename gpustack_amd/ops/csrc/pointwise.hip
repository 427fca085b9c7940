// Pointwise / memory-bound serving kernels for MI355X (gfx950).
//
// Replaces the elementwise+norm ops the reference's external engines supply
// (survey: SURVEY.md §2.9 #1 — engine kernels: RMSNorm, RoPE, activation,
// KV-cache scatter, sampling). All kernels are HBM-bound: bf16 IO is
// vectorized as u16x8 (16 B/lane), accumulation in f32, grid-stride loops
// capped so the scheduler keeps ~8 blocks/CU in flight.
#include "common.h"

// ---------------------------------------------------------------------------
// RMSNorm: out[t, :] = x[t, :] / rms(x[t, :]) * w   (row-parallel, 1 block/row)
// H <= 8192 keeps the row in registers (256 thr * 4 * u16x8); larger H
// re-reads through L2.
// ---------------------------------------------------------------------------
namespace {

constexpr int NORM_THREADS = 256;
constexpr int NORM_MAX_VEC = 4; // u16x8 per thread held in registers

// tokens (or null): `in` is a table of `vocab` rows, row t the one of tokens[t],
// which `rows` gets as well. That is the embedding and the first norm in a launch:
// 16 rows of 4096 12.5 + 4.6 -> 5.1 us, 48 4.7 + 4.7 -> 5.1. The caller refuses
// tokens out of range (ForwardMeta.checked); here they only read nothing outside
// the table and make a row of zeros.
__global__ void rms_norm_kernel(unsigned short* __restrict__ out,
                                const unsigned short* __restrict__ in,
                                const unsigned short* __restrict__ w,
                                const long* __restrict__ tokens,
                                unsigned short* __restrict__ rows, long vocab,
                                float eps, int T, int H) {
  const int nvec = H / 8; // H % 8 == 0 enforced on host
  const bool cached = nvec <= NORM_THREADS * NORM_MAX_VEC;
  for (int row = blockIdx.x; row < T; row += gridDim.x) {
    const unsigned short* rp = in + (long)row * H;
    if (tokens != nullptr) {
      const long id = tokens[row];
      unsigned short* to = rows + (long)row * H;
      rp = in + id * H;
      if (id < 0 || id >= vocab) {           // the same for the workgroup
        const u16x8 none = {0, 0, 0, 0, 0, 0, 0, 0};
        for (int v = threadIdx.x; v < nvec; v += NORM_THREADS) {
          *reinterpret_cast<u16x8*>(to + v * 8) = none;
          *reinterpret_cast<u16x8*>(out + (long)row * H + v * 8) = none;
        }
        continue;
      }
    }
    // in registers, all loads before the first use, with the weights (embedding and
    // norm, us: one row of 4096 2.9 -> 2.0, 48 3.4 -> 2.4, 512 4.7 -> 3.9)
    u16x8 vals[NORM_MAX_VEC], wv[NORM_MAX_VEC];
    float ss = 0.f;
    auto add = [&](const u16x8 u, int v) {
      if (tokens != nullptr)
        *reinterpret_cast<u16x8*>(rows + (long)row * H + v * 8) = u;
      float f[8];
      bf8_to_f32(u, f);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = __builtin_fmaf(f[i], f[i], ss);
    };
    if (cached) {
#pragma unroll
      for (int slot = 0; slot < NORM_MAX_VEC; ++slot) {
        const int v = threadIdx.x + slot * NORM_THREADS;
        if (v >= nvec) break;
        vals[slot] = *reinterpret_cast<const u16x8*>(rp + v * 8);
        wv[slot] = *reinterpret_cast<const u16x8*>(w + v * 8);
      }
#pragma unroll
      for (int slot = 0; slot < NORM_MAX_VEC; ++slot) {
        const int v = threadIdx.x + slot * NORM_THREADS;
        if (v >= nvec) break;
        add(vals[slot], v);
      }
    } else {
      for (int v = threadIdx.x; v < nvec; v += NORM_THREADS)
        add(*reinterpret_cast<const u16x8*>(rp + v * 8), v);
    }
    // block reduce: wave reduce + LDS
    __shared__ float red[NORM_THREADS / WAVE_SIZE];
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & (WAVE_SIZE - 1)) == 0) red[threadIdx.x / WAVE_SIZE] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < NORM_THREADS / WAVE_SIZE; ++i) tot += red[i];
    const float inv = rsqrtf(tot / H + eps);
    unsigned short* op = out + (long)row * H;
    auto put = [&](const u16x8 u, const u16x8 g, int v) {
      float f[8], o[8];
      bf8_to_f32(u, f);
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = f[i] * inv * bf2f(g[i]);
      *reinterpret_cast<u16x8*>(op + v * 8) = f32_to_bf8(o);
    };
    if (cached) {
#pragma unroll
      for (int slot = 0; slot < NORM_MAX_VEC; ++slot) {
        const int v = threadIdx.x + slot * NORM_THREADS;
        if (v >= nvec) break;
        put(vals[slot], wv[slot], v);
      }
    } else {
      for (int v = threadIdx.x; v < nvec; v += NORM_THREADS)
        put(*reinterpret_cast<const u16x8*>(rp + v * 8),
            *reinterpret_cast<const u16x8*>(w + v * 8), v);
    }
    __syncthreads();
  }
}

// residual += x ; x = rmsnorm(residual) * w      (both updated in place)
// PARTS: x is only written; what is added comes as the fp32 parts [parts, N, H]
// of a product cut over k, rounded as its join would. That saves the join's
// launch: 48 rows of 4096 in four parts 4.6 + 4.7 us -> 5.6.
// CHOSEN: the same for the bf16 rows [N, parts, H] of a row's experts, added up in
// fp32 and rounded as their sum would be: 64 rows of 2048 from 8 experts 5.0 + 4.8
// us -> 5.4, 4068 rows 27 + 15 -> 34 (5.3 TB/s).
// pick (or null): row t is the norm of row pick[t] of N, the result goes to `out`
// and the sum nowhere: the last norm, of the rows whose logits are asked for. That
// saves the gather behind it (4.7 us). Picks out of range, which the caller
// refuses, are clamped.
enum NormFrom { ROWS, PARTS, CHOSEN };

template <int FROM>
DEVICE_INLINE u16x8 norm_addend(const unsigned short* x, const void* from,
                                long row, int v, int parts, int N, int H) {
  if constexpr (FROM == PARTS)
    return join_parts8((const float*)from + row * H + v * 8, (long)N * H, parts);
  else if constexpr (FROM == CHOSEN)
    return sum_rows8((const unsigned short*)from + row * parts * H + v * 8, H,
                     parts);
  else
    return *reinterpret_cast<const u16x8*>(x + row * H + v * 8);
}

template <int FROM, int THREADS>
__global__ __launch_bounds__(THREADS) void fused_add_rms_norm_kernel(unsigned short* out,
                                          const unsigned short* x,
                                          unsigned short* __restrict__ residual,
                                          const unsigned short* __restrict__ w,
                                          const void* __restrict__ from,
                                          const long* __restrict__ pick,
                                          int parts, float eps, int T, int N,
                                          int H) {
  const int nvec = H / 8;
  // Rows of more than 8192 read the rounded sum back, with 512 threads too, which
  // could hold it: else a row's rounding would depend on the rows beside it.
  const bool cached = nvec <= NORM_THREADS * NORM_MAX_VEC;
  constexpr int SLOTS = NORM_THREADS * NORM_MAX_VEC / THREADS;
  for (int row = blockIdx.x; row < T; row += gridDim.x) {
    long src = row;
    if (pick != nullptr) {
      src = pick[row];
      if (src < 0) src += N;
      src = src < 0 ? 0 : src < N ? src : N - 1;
    }
    unsigned short* op = out + (long)row * H;
    unsigned short* rp = residual + src * H;
    // up to SLOTS chunks of 8 a thread in registers, and the weights, which come with
    // them and not behind the sum (that, the wave's sum without the LDS and eight parts
    // in flight, us a launch behind the writer of the parts: one row of 4096 in 4 parts
    // 2.9 -> 2.6, in 8 3.7 -> 3.4, 48 rows 4.4 -> 4.1 and 6.3 -> 6.2)
    // Squares are multiply-adds by name: of a sum that begins with a constant 0 the
    // compiler may round the second one first, and a row in a few hundred is another.
    float vals[SLOTS][8];
    u16x8 wv[SLOTS];
    float ss = 0.f;
    if (cached) {
#pragma unroll
      for (int slot = 0; slot < SLOTS; ++slot) {
        const int v = threadIdx.x + slot * THREADS;
        if (v >= nvec) break;
        const u16x8 ur = *reinterpret_cast<const u16x8*>(rp + v * 8);
        wv[slot] = *reinterpret_cast<const u16x8*>(w + v * 8);
        const u16x8 ux = norm_addend<FROM>(x, from, src, v, parts, N, H);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          vals[slot][i] = bf2f(ux[i]) + bf2f(ur[i]);
          ss = __builtin_fmaf(vals[slot][i], vals[slot][i], ss);
        }
        if (pick == nullptr)
          *reinterpret_cast<u16x8*>(rp + v * 8) = f32_to_bf8(vals[slot]);
      }
    } else {
      for (int v = threadIdx.x; v < nvec; v += THREADS) {
        u16x8 ur = *reinterpret_cast<const u16x8*>(rp + v * 8);
        const u16x8 ux = norm_addend<FROM>(x, from, src, v, parts, N, H);
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          f[i] = bf2f(ux[i]) + bf2f(ur[i]);
          ss = __builtin_fmaf(f[i], f[i], ss);
        }
        if (pick == nullptr)
          *reinterpret_cast<u16x8*>(rp + v * 8) = f32_to_bf8(f);
      }
    }
    __shared__ float red[THREADS / WAVE_SIZE];
    ss = wave_reduce_sum(ss);
    if ((threadIdx.x & (WAVE_SIZE - 1)) == 0) red[threadIdx.x / WAVE_SIZE] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < THREADS / WAVE_SIZE; ++i) tot += red[i];
    const float inv = rsqrtf(tot / H + eps);
    if (cached) {
#pragma unroll
      for (int slot = 0; slot < SLOTS; ++slot) {
        const int v = threadIdx.x + slot * THREADS;
        if (v >= nvec) break;
        float o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = vals[slot][i] * inv * bf2f(wv[slot][i]);
        *reinterpret_cast<u16x8*>(op + v * 8) = f32_to_bf8(o);
      }
    } else {
      for (int v = threadIdx.x; v < nvec; v += THREADS) {
        // residual now holds the sum (bf16-rounded); re-read it.
        float f[8];
        u16x8 u = *reinterpret_cast<const u16x8*>(rp + v * 8);
        bf8_to_f32(u, f);
        if (pick != nullptr) {               // add again, and round like that
          const u16x8 ux = norm_addend<FROM>(x, from, src, v, parts, N, H);
#pragma unroll
          for (int i = 0; i < 8; ++i) f[i] += bf2f(ux[i]);
          bf8_to_f32(f32_to_bf8(f), f);
        }
        u16x8 wv8 = *reinterpret_cast<const u16x8*>(w + v * 8);
        float o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = f[i] * inv * bf2f(wv8[i]);
        *reinterpret_cast<u16x8*>(op + v * 8) = f32_to_bf8(o);
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Rotary embedding (GPT-NeoX style halves), in-place on q and k.
// cos_sin: [max_pos, rot_dim] f32, first rot_dim/2 cos then rot_dim/2 sin,
// precomputed on host (Appendix B: no on-device trig).
// Work unit: one (token, head, 8-dim chunk of the first half).
// ---------------------------------------------------------------------------
__global__ void rope_neox_kernel(const long* __restrict__ positions,
                                 unsigned short* __restrict__ q,
                                 unsigned short* __restrict__ k,
                                 const float* __restrict__ cos_sin,
                                 int T, int Hq, int Hk, int D, int R,
                                 long qs, long ks) {  // row strides (elements)
  const int half = R / 2;
  const int chunks_per_head = half / 8; // R/2 % 8 == 0 enforced on host
  const long total = (long)T * (Hq + Hk) * chunks_per_head;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int c = idx % chunks_per_head;
    const int h = (idx / chunks_per_head) % (Hq + Hk);
    const int t = idx / ((long)chunks_per_head * (Hq + Hk));
    const long pos = positions[t];
    const float* cs = cos_sin + pos * R + c * 8;
    unsigned short* base =
        (h < Hq) ? q + (long)t * qs + (long)h * D
                 : k + (long)t * ks + (long)(h - Hq) * D;
    u16x8 u1 = *reinterpret_cast<const u16x8*>(base + c * 8);
    u16x8 u2 = *reinterpret_cast<const u16x8*>(base + half + c * 8);
    float o1[8], o2[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x1 = bf2f(u1[i]), x2 = bf2f(u2[i]);
      const float co = cs[i], si = cs[half + i];
      o1[i] = x1 * co - x2 * si;
      o2[i] = x2 * co + x1 * si;
    }
    *reinterpret_cast<u16x8*>(base + c * 8) = f32_to_bf8(o1);
    *reinterpret_cast<u16x8*>(base + half + c * 8) = f32_to_bf8(o2);
  }
}

// ---------------------------------------------------------------------------
// SiLU-and-mul: out[t, i] = silu(x[t, i]) * x[t, I + i]
// ---------------------------------------------------------------------------
__global__ void silu_and_mul_kernel(unsigned short* __restrict__ out,
                                    const unsigned short* __restrict__ x,
                                    long T, int I) {
  const long total = T * (I / 8);
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const long t = idx / (I / 8);
    const int c = idx % (I / 8);
    const unsigned short* g = x + t * 2 * I + c * 8;
    const unsigned short* u = x + t * 2 * I + I + c * 8;
    u16x8 gv = *reinterpret_cast<const u16x8*>(g);
    u16x8 uv = *reinterpret_cast<const u16x8*>(u);
    float o[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float a = bf2f(gv[i]);
      o[i] = a / (1.f + __expf(-a)) * bf2f(uv[i]);
    }
    *reinterpret_cast<u16x8*>(out + t * I + c * 8) = f32_to_bf8(o);
  }
}

// ---------------------------------------------------------------------------
// reshape_and_cache: scatter fresh per-token K/V into the paged pool.
// k/v: [T, Hkv, D] bf16 ; caches: [num_blocks, Hkv, BS, D] ; slot[t] = global
// slot index (block*BS + offset), -1 = skip.
// ---------------------------------------------------------------------------
__global__ void reshape_and_cache_fp8_kernel(const unsigned short* __restrict__ k,
                                             const unsigned short* __restrict__ v,
                                             unsigned char* __restrict__ kc,
                                             unsigned char* __restrict__ vc,
                                             const long* __restrict__ slots,
                                             int T, int Hkv, int D, int BS,
                                             long ks, long vs) {
  const int chunks = D / 8;
  const long total = (long)T * Hkv * chunks;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int c = idx % chunks;
    const int h = (idx / chunks) % Hkv;
    const int t = idx / ((long)chunks * Hkv);
    const long slot = slots[t];
    if (slot < 0) continue;
    const long blk = slot / BS, off = slot % BS;
    const long dst = ((blk * Hkv + h) * BS + off) * D + c * 8;
    const long hoff = (long)h * D + c * 8;
    u16x8 kv8 = *reinterpret_cast<const u16x8*>(k + (long)t * ks + hoff);
    u16x8 vv8 = *reinterpret_cast<const u16x8*>(v + (long)t * vs + hoff);
    u8x8 ko, vo;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      ko[i] = f32_to_fp8(bf2f(kv8[i]));
      vo[i] = f32_to_fp8(bf2f(vv8[i]));
    }
    *reinterpret_cast<u8x8*>(kc + dst) = ko;
    *reinterpret_cast<u8x8*>(vc + dst) = vo;
  }
}

__global__ void reshape_and_cache_kernel(const unsigned short* __restrict__ k,
                                         const unsigned short* __restrict__ v,
                                         unsigned short* __restrict__ kc,
                                         unsigned short* __restrict__ vc,
                                         const long* __restrict__ slots,
                                         int T, int Hkv, int D, int BS,
                                         long ks, long vs) {
  const int chunks = D / 8;
  const long total = (long)T * Hkv * chunks;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int c = idx % chunks;
    const int h = (idx / chunks) % Hkv;
    const int t = idx / ((long)chunks * Hkv);
    const long slot = slots[t];
    if (slot < 0) continue;
    const long blk = slot / BS, off = slot % BS;
    const long dst = ((blk * Hkv + h) * BS + off) * D + c * 8;
    const long hoff = (long)h * D + c * 8;
    *reinterpret_cast<u16x8*>(kc + dst) =
        *reinterpret_cast<const u16x8*>(k + (long)t * ks + hoff);
    *reinterpret_cast<u16x8*>(vc + dst) =
        *reinterpret_cast<const u16x8*>(v + (long)t * vs + hoff);
  }
}

// ---------------------------------------------------------------------------
// The way from a fused q|k|v projection row to attention in one launch:
// optional RMS norm of every q and k head (one weight vector each), rotation
// of q and k in place (halves), keys and values to their cache slots (-1 =
// skip). LPH = D / 16 lanes share a head: a lane holds 8 channels of the first
// half and the 8 that they rotate with, so the pair is in its registers and
// the norm takes log2(LPH) cross-lane steps. Bound by the row's bytes; two
// norms, three copies, rotation and cache write as launches of their own took
// 170 us a layer at 4068 rows of 32 + 2 x 4 heads (a workgroup per head).
// ---------------------------------------------------------------------------
// PARTS: the row comes as fp32 parts [parts, T, (Hq + 2 Hk) * D] of a product
// cut over k and is written here (48 rows of 32 + 2 x 8 heads in five parts 4.5 +
// 4.7 us -> 6.0).
template <int LPH, bool FP8, bool PARTS>
__global__ __launch_bounds__(256) void qkv_store_kernel(
    unsigned short* __restrict__ qkv,          // [T, (Hq + 2 Hk) * D]
    const float* __restrict__ from, int parts,
    const unsigned short* __restrict__ qw,     // [D] or null
    const unsigned short* __restrict__ kw,     // [D] or null
    const float* __restrict__ cos_sin,         // [positions, D]
    const long* __restrict__ positions, const long* __restrict__ slots,
    void* __restrict__ kc, void* __restrict__ vc,  // [nb, Hk, BS, D]
    long heads, int Hq, int Hk, int BS, float eps) {
  constexpr int D = LPH * 16, HALF = D / 2;
  const int H = Hq + 2 * Hk;
  const int c = threadIdx.x % LPH * 8;
  const long step = (long)gridDim.x * (256 / LPH);
  for (long u = (long)blockIdx.x * (256 / LPH) + threadIdx.x / LPH; u < heads;
       u += step) {
    const long t = u / H;
    const int h = (int)(u % H);
    unsigned short* p = qkv + u * D + c;
    // what hangs on the row's place is asked for in front of the row
    const float* cs = cos_sin + positions[t] * D + c;
    const long slot = h < Hq ? -1 : slots[t];
    float co[8], si[8];
    if (h < Hq + Hk) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        co[i] = cs[i];
        si[i] = cs[HALF + i];
      }
    }
    u16x8 a, b;
    if constexpr (PARTS) {
      a = join_parts8(from + u * D + c, heads * D, parts);
      b = join_parts8(from + u * D + c + HALF, heads * D, parts);
      if (h >= Hq + Hk) {
        *reinterpret_cast<u16x8*>(p) = a;
        *reinterpret_cast<u16x8*>(p + HALF) = b;
      }
    } else {
      a = *reinterpret_cast<const u16x8*>(p);
      b = *reinterpret_cast<const u16x8*>(p + HALF);
    }
    if (h < Hq + Hk) {
      float x[8], y[8], o[8];
      bf8_to_f32(a, x);
      bf8_to_f32(b, y);
      const unsigned short* w = h < Hq ? qw : kw;
      if (w != nullptr) {
        float ss = 0.f, wx[8], wy[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += x[i] * x[i] + y[i] * y[i];
#pragma unroll
        for (int m = LPH / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
        const float inv = rsqrtf(ss / D + eps);
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
      *reinterpret_cast<u16x8*>(p) = a;
      *reinterpret_cast<u16x8*>(p + HALF) = b;
    }
    if (h < Hq || slot < 0) continue;
    const int g = (h - Hq) % Hk;
    const long dst = ((slot / BS * Hk + g) * BS + slot % BS) * D + c;
    void* pool = h < Hq + Hk ? kc : vc;
    if constexpr (FP8) {
      u8x8 qa, qb;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        qa[i] = f32_to_fp8(bf2f(a[i]));
        qb[i] = f32_to_fp8(bf2f(b[i]));
      }
      *reinterpret_cast<u8x8*>((unsigned char*)pool + dst) = qa;
      *reinterpret_cast<u8x8*>((unsigned char*)pool + dst + HALF) = qb;
    } else {
      *reinterpret_cast<u16x8*>((unsigned short*)pool + dst) = a;
      *reinterpret_cast<u16x8*>((unsigned short*)pool + dst + HALF) = b;
    }
  }
}

// ---------------------------------------------------------------------------
// Greedy sampling: argmax over vocab per row (ties -> lowest index).
// One block per row: 16 waves with four 16-byte loads in flight each, the
// maximum of eight values first and its place only where it counts. Bound by
// how fast one CU takes a row in and compares it (256 KB of a 128256-word
// vocabulary): one row 8.1 us, 16 8.6, 64 8.8, 300 17. With eight loads in flight,
// the last ones once more behind the end, these take 7.6, 8.0, 8.2 and 17.1, but
// 64 rows of 4096 words 3.9 for 3.1, of 151936 10.1 for 9.5, 300 of 32001 10.4 for 8.6.
// The words are also left in `host` (pinned memory, or null), which saves a copy
// behind the kernel.
// ---------------------------------------------------------------------------
constexpr int GS_THREADS = 1024;

__global__ __launch_bounds__(GS_THREADS) void greedy_sample_kernel(
    long* __restrict__ out, long* __restrict__ host,
    const unsigned short* __restrict__ logits, int N, int V) {
  const int row = blockIdx.x;
  if (row >= N) return;
  const unsigned short* rp = logits + (long)row * V;
  float best = -INFINITY;
  int besti = 0x7fffffff;              // first index of `best` seen so far
  const int nvec = V / 8;
  auto take = [&](const u16x8 u, int v) {
    float f[8], mx;
    bf8_to_f32(u, f);
    mx = fmaxf(fmaxf(fmaxf(f[0], f[1]), fmaxf(f[2], f[3])),
               fmaxf(fmaxf(f[4], f[5]), fmaxf(f[6], f[7])));
    if (mx > best) {                   // a thread's indices only grow
      best = mx;
      int i = 7;
#pragma unroll
      for (int j = 6; j >= 0; --j) i = f[j] == mx ? j : i;
      besti = v * 8 + i;
    }
  };
  int v = threadIdx.x;
  for (; v + 3 * GS_THREADS < nvec; v += 4 * GS_THREADS) {
    u16x8 u[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      u[j] = *reinterpret_cast<const u16x8*>(rp + (v + j * GS_THREADS) * 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) take(u[j], v + j * GS_THREADS);
  }
  for (; v < nvec; v += GS_THREADS)
    take(*reinterpret_cast<const u16x8*>(rp + v * 8), v);
  for (int gi = nvec * 8 + threadIdx.x; gi < V; gi += GS_THREADS) {
    const float f = bf2f(rp[gi]);
    if (f > best) { best = f; besti = gi; }
  }
  // wave reduce, then LDS reduce
  auto join = [&](int from) {
#pragma unroll
    for (int m = from; m >= 1; m >>= 1) {
      const float ov = __shfl_xor(best, m, WAVE_SIZE);
      const int oi = __shfl_xor(besti, m, WAVE_SIZE);
      if (ov > best || (ov == best && oi < besti)) { best = ov; besti = oi; }
    }
  };
  join(32);
  __shared__ float sv[GS_THREADS / WAVE_SIZE];
  __shared__ int si[GS_THREADS / WAVE_SIZE];
  const int wid = threadIdx.x / WAVE_SIZE;
  if ((threadIdx.x & (WAVE_SIZE - 1)) == 0) { sv[wid] = best; si[wid] = besti; }
  __syncthreads();
  if (threadIdx.x < GS_THREADS / WAVE_SIZE) {
    best = sv[threadIdx.x];
    besti = si[threadIdx.x];
    join(GS_THREADS / WAVE_SIZE / 2);
    // a row without any number (all NaN) still names a word
    if (threadIdx.x == 0) {
      const long word = besti == 0x7fffffff ? 0 : besti;
      out[row] = word;
      if (host != nullptr) host[row] = word;
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Launchers (called from bindings.cpp)
// ---------------------------------------------------------------------------
static inline int pw_grid(long total_threads_needed, int block) {
  long blocks = (total_threads_needed + block - 1) / block;
  if (blocks > 2048) blocks = 2048; // ~8 blocks/CU, grid-stride the rest
  if (blocks < 1) blocks = 1;
  return (int)blocks;
}

// tokens: null, or the rows of `in` [vocab, H] that `rows` gets
void rms_norm_launch(void* out, const void* in, const void* w,
                     const long* tokens, void* rows, long vocab, float eps,
                     int T, int H, hipStream_t s) {
  int grid = T < 8192 ? (T < 1 ? 1 : T) : 8192;
  hipLaunchKernelGGL(rms_norm_kernel, dim3(grid), dim3(NORM_THREADS), 0, s,
                     (unsigned short*)out, (const unsigned short*)in,
                     (const unsigned short*)w, tokens, (unsigned short*)rows,
                     vocab, eps, T, H);
}

namespace {
template <int THREADS>
void norm_launch(void* out, const void* x, void* residual, const void* w,
                 const void* from, int chosen, const long* pick, int parts,
                 float eps, int T, int N, int H, hipStream_t s) {
  int grid = T < 8192 ? (T < 1 ? 1 : T) : 8192;
  hipLaunchKernelGGL(
      (from == nullptr ? fused_add_rms_norm_kernel<ROWS, THREADS>
       : chosen        ? fused_add_rms_norm_kernel<CHOSEN, THREADS>
                       : fused_add_rms_norm_kernel<PARTS, THREADS>),
      dim3(grid), dim3(THREADS), 0, s, (unsigned short*)out,
      (const unsigned short*)x, (unsigned short*)residual,
      (const unsigned short*)w, from, pick, parts, eps, T, N, H);
}
}  // namespace

// out [T, H], x and residual [N, H]. from: null, or what is added instead of x:
// fp32 parts [parts, N, H] or, with chosen, bf16 rows [N, parts, H]. pick: null
// (T = N), or the rows that out has.
void fused_add_rms_norm_launch(void* out, const void* x, void* residual,
                               const void* w, const void* from, int chosen,
                               const long* pick, int parts, float eps, int T,
                               int N, int H, hipStream_t s) {
  // Few rows of more than 2048: 512 threads, one chunk of 8 a thread up to 4096,
  // for the latency of a row's loads (us back to back, 256 -> 512 threads: 16 rows
  // of 4096 3.4 -> 2.8, in 8 parts 4.9 -> 3.8, of 8192 4.8 -> 3.7 and 7.6 -> 5.6;
  // 512 rows of 4096 4.7 -> 4.5); more rows fill the CUs with 256.
  if (T <= 512 && H > 2048)
    norm_launch<512>(out, x, residual, w, from, chosen, pick, parts, eps, T, N, H,
                     s);
  else
    norm_launch<NORM_THREADS>(out, x, residual, w, from, chosen, pick, parts, eps,
                              T, N, H, s);
}

void rope_neox_launch(const long* positions, void* q, void* k,
                      const float* cos_sin, int T, int Hq, int Hk, int D,
                      int R, long qs, long ks, hipStream_t s) {
  long total = (long)T * (Hq + Hk) * (R / 2 / 8);
  hipLaunchKernelGGL(rope_neox_kernel, dim3(pw_grid(total, 256)), dim3(256), 0,
                     s, positions, (unsigned short*)q, (unsigned short*)k,
                     cos_sin, T, Hq, Hk, D, R, qs, ks);
}

void silu_and_mul_launch(void* out, const void* x, long T, int I,
                         hipStream_t s) {
  long total = T * (I / 8);
  hipLaunchKernelGGL(silu_and_mul_kernel, dim3(pw_grid(total, 256)), dim3(256),
                     0, s, (unsigned short*)out, (const unsigned short*)x, T, I);
}

void reshape_and_cache_launch(const void* k, const void* v, void* kc, void* vc,
                              const long* slots, int T, int Hkv, int D, int BS,
                              long ks, long vs, int fp8, hipStream_t s) {
  long total = (long)T * Hkv * (D / 8);
  if (fp8) {
    hipLaunchKernelGGL(reshape_and_cache_fp8_kernel, dim3(pw_grid(total, 256)),
                       dim3(256), 0, s, (const unsigned short*)k,
                       (const unsigned short*)v, (unsigned char*)kc,
                       (unsigned char*)vc, slots, T, Hkv, D, BS, ks, vs);
  } else {
    hipLaunchKernelGGL(reshape_and_cache_kernel, dim3(pw_grid(total, 256)),
                       dim3(256), 0, s, (const unsigned short*)k,
                       (const unsigned short*)v, (unsigned short*)kc,
                       (unsigned short*)vc, slots, T, Hkv, D, BS, ks, vs);
  }
}

void greedy_sample_launch(long* out, long* host, const void* logits, int N, int V,
                          hipStream_t s) {
  if (N == 0) return;
  hipLaunchKernelGGL(greedy_sample_kernel, dim3(N), dim3(GS_THREADS), 0, s, out,
                     host, (const unsigned short*)logits, N, V);
}

void qkv_store_launch(void* qkv, const float* from, int parts, const void* qw,
                      const void* kw,
                      const float* cos_sin, const long* positions,
                      const long* slots, void* kc, void* vc, long T, int Hq,
                      int Hk, int D, int BS, float eps, int fp8,
                      int* err_unsupported, hipStream_t s) {
  *err_unsupported = D != 64 && D != 128 && D != 256;
  const long heads = T * (Hq + 2 * Hk);
  if (*err_unsupported || heads == 0) return;
  const long per = 256 / (D / 16);
  const long blocks = (heads + per - 1) / per;
  const unsigned grid = (unsigned)(blocks > 16384 ? 16384 : blocks);
#define QKV(L, F)                                                             \
  hipLaunchKernelGGL((from != nullptr ? qkv_store_kernel<L, F, true>          \
                                      : qkv_store_kernel<L, F, false>),       \
                     dim3(grid), dim3(256), 0, s, (unsigned short*)qkv, from, \
                     parts, (const unsigned short*)qw,                        \
                     (const unsigned short*)kw, cos_sin, positions, slots,    \
                     kc, vc, heads, Hq, Hk, BS, eps)
  if (D == 64) {
    if (fp8) QKV(4, true);
    else QKV(4, false);
  } else if (D == 128) {
    if (fp8) QKV(8, true);
    else QKV(8, false);
  } else {
    if (fp8) QKV(16, true);
    else QKV(16, false);
  }
#undef QKV
}
