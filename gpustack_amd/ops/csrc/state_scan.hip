// Recurrent mixers with one matrix state per head and sequence (gfx950).
//
//   S_t = a_t S_(t-1) + b_t k_t v_t^T,    y_t = S_t^T q_t + skip * v_t
//
// S [N x P] is fp32 and lives in the sequence's slot of a state pool
// [slots, H, N, P]. A batch is ragged: sequence s brings rows seq_first[s]
// .. seq_first[s] + seq_rows[s] - 1 (a prompt portion, or one decoded
// token); its first row's position says whether the slot is read (> 0) or
// the state starts from zero (== 0). Every kernel here walks or indexes
// rows through that per-sequence view, so a prompt cut anywhere, a decode
// row and a mixed batch give the same states.
//
//   state_scan       : the recurrence. A wave owns PL value channels of one
//                      (sequence, head); the N state rows are split over
//                      TPP lanes per channel, NR rows each, in registers.
//                      Rows are staged CH at a time through LDS (k, q, v,
//                      decay, step), then walked in order. Step sizes and
//                      decays are computed here in fp32: a = exp(-exp(A_log)
//                      * dt), b = dt = softplus(raw + bias), or constants.
//   gated_group_norm : gate (SiLU or sigmoid) and RMS norm in equal parts of
//                      the row, in either order
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

// (With expf and a division the chunks of an activated scan, 7032 rows of 16 heads of
// 128 x 128, took 262 us in both launches, and take 251.)
DEVICE_INLINE float silu_f(float z) { return over_one_plus_exp(z, z); }
DEVICE_INLINE float sigmoid_f(float z) { return over_one_plus_exp(1.f, z); }
// softplus without a switch-over: max(x, 0) + log1p(exp(-|x|))
DEVICE_INLINE float softplus_f(float x) {
  return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
}

struct ScanArgs {
  long ld_src, ld_dt;
  int col_x, col_b, col_c, col_dt;
  int H, G, N, P, act;
  const float* dt_bias;    // [H] with dt
  const float* a_log;      // [H] with dt
  const float* skip;       // [H] or null
  const float* decay;      // [H] without dt
  float* state;            // [nslots, H, N, P]
  const int* seq_first;
  const int* seq_rows;
  const int* state_slots;
  const int* pos32;
  int nslots, T;
  // sequences cut into runs of rows (state_chunk_kernel), or null
  const int* runs;         // [nruns, 4] first row, rows, sequence, the list
                           // index of the sequence's first run
  int nruns, nseq;
  int ncut;                // runs in front of the list that have places below;
                           // only sequences of one run may lie behind them
  float* ends;             // [ncut, H, N, P] state behind a run
  float* scratch;          // [ncut, H, N, P]
  float* falls;            // [ncut, H] product of a run's decays
};

constexpr int CH = 16;     // rows staged per pass

// One wave per (sequence, head, block of PL = 64 / TPP value channels).
// lane = ns * PL + pl: channel p0 + pl, state rows n = r * TPP + ns. CHG rows
// are staged per pass (fewer for the widest states, to fit the LDS).
template <typename TS, typename TD, int NR, int TPP, int CHG>
__global__ __launch_bounds__(64) void state_scan_kernel(
    float* __restrict__ y, const TS* __restrict__ src,
    const TD* __restrict__ dt_src, ScanArgs p) {
  constexpr int PL = 64 / TPP;
  constexpr int NP = NR * TPP;               // padded state rows
  __shared__ float ks[CHG][NP];
  __shared__ float qs[CHG][NP];
  __shared__ float vs[CHG][PL];
  __shared__ float a_s[CHG], b_s[CHG];
  const int s = blockIdx.x, h = blockIdx.y, p0 = blockIdx.z * PL;
  const int lane = threadIdx.x;
  const int pl = lane % PL, ns = lane / PL;
  const int first = p.seq_first[s], n = p.seq_rows[s];
  if (first < 0 || n < 1 || first + n > p.T) return;
  const int slot = min(max(p.state_slots[s], 0), p.nslots - 1);
  const int hist = p.pos32[first];
  const int N = p.N, P = p.P;
  const int g = h / (p.H / p.G);
  const int pc = p0 + pl;
  const bool live = pc < P;
  float* sp = p.state + ((long)slot * p.H + h) * N * P;
  float S[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int nn = r * TPP + ns;
    S[r] = (hist > 0 && live && nn < N) ? sp[(long)nn * P + pc] : 0.f;
  }
  const float skip = p.skip != nullptr ? p.skip[h] : 0.f;
  const float a_rate = dt_src != nullptr ? expf(p.a_log[h]) : 0.f;
  const float dtb = dt_src != nullptr ? p.dt_bias[h] : 0.f;
  const float a_const = dt_src == nullptr ? p.decay[h] : 0.f;

  for (int c0 = 0; c0 < n; c0 += CHG) {
    const int rows = min(CHG, n - c0);
    __syncthreads();
    for (int i = lane; i < rows * NP; i += 64) {
      const int r = i / NP, nn = i % NP;
      float kv = 0.f, qv = 0.f;
      if (nn < N) {
        const TS* rp = src + (long)(first + c0 + r) * p.ld_src;
        kv = ld(rp + p.col_b + g * N + nn);
        qv = ld(rp + p.col_c + g * N + nn);
        if (p.act) { kv = silu_f(kv); qv = silu_f(qv); }
      }
      ks[r][nn] = kv;
      qs[r][nn] = qv;
    }
    for (int i = lane; i < rows * PL; i += 64) {
      const int r = i / PL, c = i % PL;
      float v = 0.f;
      if (p0 + c < P) {
        v = ld(src + (long)(first + c0 + r) * p.ld_src + p.col_x + h * P + p0 + c);
        if (p.act) v = silu_f(v);
      }
      vs[r][c] = v;
    }
    if (lane < rows) {
      if (dt_src != nullptr) {
        const float dt = softplus_f(
            ld(dt_src + (long)(first + c0 + lane) * p.ld_dt + p.col_dt + h) + dtb);
        a_s[lane] = expf(-a_rate * dt);
        b_s[lane] = dt;
      } else {
        a_s[lane] = a_const;
        b_s[lane] = 1.f;
      }
    }
    __syncthreads();
    for (int r = 0; r < rows; ++r) {
      const float a = a_s[r];
      const float v = vs[r][pl];
      const float bv = b_s[r] * v;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < NR; ++j) {
        const int nn = j * TPP + ns;
        S[j] = a * S[j] + ks[r][nn] * bv;
        acc += S[j] * qs[r][nn];
      }
#pragma unroll
      for (int m = PL; m < 64; m <<= 1) acc += __shfl_xor(acc, m, WAVE_SIZE);
      if (ns == 0 && live)
        y[(long)(first + c0 + r) * p.H * P + h * P + pc] = acc + skip * v;
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const int nn = r * TPP + ns;
    if (live && nn < N) sp[(long)nn * P + pc] = S[r];
  }
}


// The same recurrence for bf16 sources whose sizes and columns are multiples
// of 8: four waves share one (sequence, head) and 4 * PL value channels, so
// k and q are staged once for all of them with 16-byte loads; the next
// CH rows are fetched into registers while the current ones are walked
// (two LDS buffers, one barrier per pass). A lane owns the state rows
// ns * NR .. ns * NR + NR - 1 and reads its k / q slice from LDS in 16-byte
// pieces; slices of different ns sit NR + 4 floats apart, on other banks.
template <int NR, int TPP>
__global__ __launch_bounds__(256) void state_scan_vec_kernel(
    float* __restrict__ y, const unsigned short* __restrict__ src,
    const unsigned short* __restrict__ dt_src, ScanArgs p) {
  constexpr int PL = 64 / TPP;
  constexpr int NP = NR * TPP;
  constexpr int NS = NR + 4;                 // floats between two ns slices
  constexpr int ROW = TPP * NS;              // floats per staged k / q row
  constexpr int PB = 4 * PL;                 // value channels per workgroup
  constexpr int KV = (CH * NP / 8 + 255) / 256;   // 16-byte loads per lane
  constexpr int VV = (CH * PB / 8 + 255) / 256;
  __shared__ __attribute__((aligned(16))) float ks[2][CH][ROW];
  __shared__ __attribute__((aligned(16))) float qs[2][CH][ROW];
  __shared__ float vs[2][CH][PB];
  __shared__ float a_s[2][CH], b_s[2][CH];
  const int s = blockIdx.x, h = blockIdx.y, pb0 = blockIdx.z * PB;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int pl = lane % PL, ns = lane / PL;
  const int first = p.seq_first[s], n = p.seq_rows[s];
  if (first < 0 || n < 1 || first + n > p.T) return;
  const int slot = min(max(p.state_slots[s], 0), p.nslots - 1);
  const int hist = p.pos32[first];
  const int N = p.N, P = p.P;
  const int g = h / (p.H / p.G);
  const int pc = pb0 + wave * PL + pl;
  const bool live = pc < P;
  float* sp = p.state + ((long)slot * p.H + h) * N * P;
  float S[NR];
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int nn = ns * NR + j;
    S[j] = (hist > 0 && live && nn < N) ? sp[(long)nn * P + pc] : 0.f;
  }
  const float skip = p.skip != nullptr ? p.skip[h] : 0.f;
  const float a_rate = dt_src != nullptr ? expf(p.a_log[h]) : 0.f;
  const float dtb = dt_src != nullptr ? p.dt_bias[h] : 0.f;
  const float a_const = dt_src == nullptr ? p.decay[h] : 0.f;
  const int nvec = N / 8;                    // 16-byte pieces per k / q row
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};

  u16x8 kreg[KV], qreg[KV], vreg[VV];
  float dreg = 0.f;
  float odd = 0.f;                           // NaN behind a value that is not finite
  auto fetch = [&](int c0) {
    const int rows = min(CH, n - c0);
#pragma unroll
    for (int u = 0; u < KV; ++u) {
      const int i = tid + u * 256;
      kreg[u] = zero8;
      qreg[u] = zero8;
      if (i < rows * nvec) {
        const int r = i / nvec, e = (i % nvec) * 8;
        const unsigned short* rp = src + (long)(first + c0 + r) * p.ld_src;
        kreg[u] = *reinterpret_cast<const u16x8*>(rp + p.col_b + g * N + e);
        qreg[u] = *reinterpret_cast<const u16x8*>(rp + p.col_c + g * N + e);
      }
    }
#pragma unroll
    for (int u = 0; u < VV; ++u) {
      const int i = tid + u * 256;
      vreg[u] = zero8;
      if (i < rows * (PB / 8)) {
        const int r = i / (PB / 8), c = (i % (PB / 8)) * 8;
        if (pb0 + c < P)
          vreg[u] = *reinterpret_cast<const u16x8*>(
              src + (long)(first + c0 + r) * p.ld_src + p.col_x + h * P + pb0 + c);
      }
    }
    if (dt_src != nullptr && tid < rows)
      dreg = bf2f(dt_src[(long)(first + c0 + tid) * p.ld_dt + p.col_dt + h]);
  };
  auto stage = [&](int buf, int c0) {
    const int rows = min(CH, n - c0);
#pragma unroll
    for (int u = 0; u < KV; ++u) {
      const int i = tid + u * 256;
      if (i < rows * nvec) {
        const int r = i / nvec, e = (i % nvec) * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          float kv = bf2f(kreg[u][k]), qv = bf2f(qreg[u][k]);
          if (p.act) { kv = silu_f(kv); qv = silu_f(qv); }
          const int nn = e + k;
          const int at = (nn / NR) * NS + nn % NR;
          ks[buf][r][at] = kv;
          qs[buf][r][at] = qv;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < VV; ++u) {
      const int i = tid + u * 256;
      if (i < rows * (PB / 8)) {
        const int r = i / (PB / 8), c = (i % (PB / 8)) * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          float v = bf2f(vreg[u][k]);
          if (p.act) v = silu_f(v);
          vs[buf][r][c + k] = v;
        }
      }
    }
    if (tid < rows) {
      if (dt_src != nullptr) {
        const float dt = softplus_f(dreg + dtb);
        a_s[buf][tid] = expf(-a_rate * dt);
        b_s[buf][tid] = dt;
      } else {
        a_s[buf][tid] = a_const;
        b_s[buf][tid] = 1.f;
      }
    }
  };
  // state rows past N (padding up to NP) keep k = q = 0: zero them once
  for (int i = tid; i < 2 * CH * ROW; i += 256) {
    (&ks[0][0][0])[i] = 0.f;
    (&qs[0][0][0])[i] = 0.f;
  }
  __syncthreads();
  fetch(0);
  int buf = 0;
  for (int c0 = 0; c0 < n; c0 += CH, buf ^= 1) {
    const int rows = min(CH, n - c0);
    stage(buf, c0);
    __syncthreads();
    if (c0 + CH < n) fetch(c0 + CH);
    const float* kb = &ks[buf][0][ns * NS];
    const float* qb = &qs[buf][0][ns * NS];
    for (int r = 0; r < rows; ++r) {
      const float a = a_s[buf][r];
      const float v = vs[buf][r][wave * PL + pl];
      const float bv = b_s[buf][r] * v;
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < NR; j += 4) {
        const f32x4 k4 = *reinterpret_cast<const f32x4*>(kb + r * ROW + j);
        const f32x4 q4 = *reinterpret_cast<const f32x4*>(qb + r * ROW + j);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          S[j + k] = a * S[j + k] + k4[k] * bv;
          acc += S[j + k] * q4[k];
        }
      }
#pragma unroll
      for (int m = PL; m < 64; m <<= 1) acc += __shfl_xor(acc, m, WAVE_SIZE);
      if (ns == 0 && live)
        y[(long)(first + c0 + r) * p.H * P + h * P + pc] = acc + skip * v;
    }
  }
#pragma unroll
  for (int j = 0; j < NR; ++j) {
    const int nn = ns * NR + j;
    if (live && nn < N) sp[(long)nn * P + pc] = S[j];
  }
}

// The same recurrence in chunks of 32 rows on the fp32 matrix instructions,
// for prompts. Inside a chunk, with c_t the sum of the logarithms of the decays
// up to row t,
//   y_t   = sum_{s <= t} e^(c_t - c_s) b_s (q_t . k_s) v_s + e^(c_t) S^T q_t
//   S_new = e^(c_31) S + sum_s e^(c_31 - c_s) b_s k_s v_s^T
// so that one chunk is four small products (Q K^T, the weighted scores times V,
// Q S, K^T V) instead of 32 dependent passes over the state. Everything stays
// fp32 (v_mfma_f32_16x16x4_f32); the c are summed in double, since their
// differences, not they, are what the weights are made of.
//   - a workgroup owns 64 value channels of one (sequence, head), a wave 16 of
//     them. Waves share q, k, v and the scores through the LDS.
//   - operands that reduce over their rows' contiguous axis are read 16 bytes
//     at a time: lane group g takes k = 4 g .. 4 g + 3 of 16, one value per
//     matrix instruction, in both operands. Rows are 4 floats longer than
//     their content, which keeps those reads off each other's banks.
//   - with that order the state, as the accumulators hold it (rows 4 g + r,
//     column l & 15), is the operand of Q S: it never leaves the registers.
//   - the next chunk's rows are fetched while this one is worked on; 48 KB.
// Bound by the chain of chunks (about 170 matrix instructions of 32 cycles a wave
// and chunk, 7.7 us). Where whole sequences leave the chip idle they are cut into
// runs of chunks (RUNS): a first launch (ENDS) works out what each run but a
// sequence's last adds to the state, from zero (the first run from the slot), and
// how far the run lets a state fall; in the second (OUTPUTS) a run's workgroup
// puts the state in front of it together from the runs before and goes through
// its rows as above. The slot is read by the first launch (the second takes the
// first run's state from `scratch`) and written by the last run in the second.
// Sequences of one run need none of that: they lie at the end of the list, without
// places, and the first launch leaves them out.
// 64 heads of 128 x 64, one sequence of 4000 rows 723 -> 266 us, six of 301 to 1900
// 433 -> 353; 16 heads of 128 x 128 918 -> 260 and 428 -> 241.
//
// EXACT: without an activation q, k and v are bf16 values, and the bf16 instructions
// multiply them as they are, at sixteen times the rate: 16 cycles for 32 k where fp32
// takes 32 for 4. The other operand (state, weighted scores, weighted v) is split into
// three bf16 parts whose sum it is to 26 bits and more, so that the products are the
// exact ones and only the sums round, in fp32 as before: error against 64 bits of y .66
// to .89 and of the state .82 to 1.00 of what the fp32 instructions leave (decays of e^-.1
// a row to ones that leave nothing), .53 and .62 (of a hundredth).
//   - the state stays in the accumulators; its parts are made a chunk, 32 rows at a time.
//   - scores are multiplied transposed, so that they lie as the operand of the product
//     with v; every wave has them all, and no barrier stands between.
//   - k and v are read down their columns (ds_read_b64_tr_b16); rows of two chunks in
//     the LDS, one barrier a chunk. Rows of q and k lie permuted, 16 bytes a lane: as two
//     reads of 8 a chunk takes 2.7 us instead of 2.1.
//   - decays and the weights e^(c_t - c_s) b_s are made for four chunks at a time, by all
//     threads: for one at a time by 32 of them a chunk takes 3.9 us.
//   - where anything is not finite its split is NaN; it shows in the rows or the state,
//     and the columns are walked again as below.
// Bound by the vector instructions (500 a wave and chunk, 72 % of the time with two
// waves a SIMD; 66 matrix ones): 64 heads of 128 x 64, whole 4000 rows 741 -> 262 us, the
// six 439 -> 165, 8 x 500 135 -> 60.
typedef __attribute__((ext_vector_type(4))) float sc_f32x4;
typedef __attribute__((ext_vector_type(2))) __bf16 sc_bf16x2;

enum ChunkPart { WHOLE, ENDS, OUTPUTS };

// An fp32 value as three bf16 ones that add up to it. PRODUCT: of products, which the
// compiler subtracts from before it rounds them (fma): up to 32 bits are left, and each
// part is the nearest to what the ones before leave. Cut, the last one lost up to an ulp,
// always towards 0, and the state of strong decays was off by 1.16 of what the fp32 form
// leaves. Values that are held are their significant bits eight by eight, which takes as
// many instructions but is the faster one (16 heads of 128 x 128, 4 x 1000 67.5 / 68.5).
struct Split8 { u32x4 part[3]; };
template <bool PRODUCT>
DEVICE_INLINE Split8 split8(const float* x) {
  Split8 s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const f32x2 v{a, b};
      const unsigned u = __builtin_bit_cast(unsigned, a);
      const unsigned w = __builtin_bit_cast(unsigned, b);
      const unsigned both =
          PRODUCT ? __builtin_bit_cast(unsigned, __builtin_convertvector(v, sc_bf16x2))
                  : __builtin_amdgcn_perm(w, u, 0x07060302u);
      s.part[part][i] = both;
      a -= __builtin_bit_cast(float, PRODUCT ? both << 16 : u & 0xffff0000u);
      b -= __builtin_bit_cast(float, (PRODUCT ? both : w) & 0xffff0000u);
    }
  }
  return s;
}
typedef __attribute__((ext_vector_type(8))) short sc_s16x8;
typedef __attribute__((ext_vector_type(4))) short sc_s16x4;
typedef __attribute__((ext_vector_type(2))) unsigned int sc_u32x2;
DEVICE_INLINE sc_f32x4 mm_bf(const u32x4 a, const u32x4 b, sc_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(sc_s16x8, a), __builtin_bit_cast(sc_s16x8, b), c, 0, 0, 0);
}
// a x the value whose parts s are, smallest first
DEVICE_INLINE sc_f32x4 mm_split(const u32x4 a, const Split8& s, sc_f32x4 c) {
  return mm_bf(a, s.part[0], mm_bf(a, s.part[1], mm_bf(a, s.part[2], c)));
}
DEVICE_INLINE sc_f32x4 mm_split(const Split8& s, const u32x4 b, sc_f32x4 c) {
  return mm_bf(s.part[0], b, mm_bf(s.part[1], b, mm_bf(s.part[2], b, c)));
}
// 16 lanes read 4 rows of 16 neighbours, a lane gets four rows of its own
DEVICE_INLINE sc_u32x2 read_down(const unsigned short* p) {
  return __builtin_bit_cast(
      sc_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) sc_s16x4*)p));
}

// EXACT: q, k and v are the bf16 values of src (no activation here).
template <int NT, int PART, bool EXACT>   // state rows / 16, padded
__global__ __launch_bounds__(256, 2) void state_chunk_kernel(
    float* __restrict__ y, const unsigned short* __restrict__ src,
    const unsigned short* __restrict__ dt_src, ScanArgs p) {
  constexpr int C = 32, NP = NT * 16, KS = NP + 4, PB = 64, VS = PB + 4;
  constexpr int KU = C * NP / 8 / 256;       // 16-byte loads of k (and q)
  static_assert(KU >= 1 && C * NP / 8 % 256 == 0, "NT is 4 or 8");
  constexpr int QR = PART == ENDS ? 1 : C;
  // fp32 rows of one chunk, or bf16 ones of two
  constexpr int F = EXACT ? 1 : C, FQ = EXACT ? 1 : QR;
  __shared__ __attribute__((aligned(16))) float qs[FQ][KS];
  __shared__ __attribute__((aligned(16))) float ks[F][KS];
  __shared__ __attribute__((aligned(16))) float vs[F][VS];
  __shared__ __attribute__((aligned(16))) float as[FQ][C + 4];
  constexpr int HS = NP + 16, WS = PB + 8, B = EXACT ? C : 1;
  __shared__ __attribute__((aligned(16))) unsigned short qh[2][EXACT ? QR : 1][HS];
  __shared__ __attribute__((aligned(16))) unsigned short kh[2][B][HS];
  __shared__ __attribute__((aligned(16))) unsigned short vh[2][B][WS];
  // decays and weights, of EXACT for SB chunks at a time
  constexpr int SB = EXACT ? 4 : 1, EB = EXACT && PART != ENDS ? SB : 1;
  // e^(c_t - c_s) b_s of row t, column s <= t
  __shared__ __attribute__((aligned(16))) float es[EB][EB > 1 ? C : 1][C + 4];
  __shared__ double cs2[SB][C];
  __shared__ float scal[SB][3][C];
  __shared__ float fell[SB];                 // EXACT: a chunk's product of decays
  double* cs = cs2[0];
  float *bl = scal[0][0], *el = scal[0][1], *wl = scal[0][2];
  int s = blockIdx.x;
  const int h = blockIdx.y, pb0 = blockIdx.z * PB;
  const int run = blockIdx.x;
  int run0 = run, first, n;
  bool ends = true;                          // the sequence ends with these rows
  if constexpr (PART == WHOLE) {
    first = p.seq_first[s];
    n = p.seq_rows[s];
  } else {
    const int* r = p.runs + (long)run * 4;
    first = r[0];
    n = r[1];
    s = r[2];
    run0 = r[3];
    if (s < 0 || s >= p.nseq || run0 < 0 || run0 > run) return;
    ends = first + n >= p.seq_first[s] + p.seq_rows[s];
    if (PART == ENDS && ends) return;
    if (run >= p.ncut && (run != run0 || !ends)) return;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lc = lane & 15, g = lane >> 4;
  if (first < 0 || n < 1 || first + n > p.T) return;
  const int slot = min(max(p.state_slots[s], 0), p.nslots - 1);
  // a state in front of these rows
  const int hist = run == run0 ? p.pos32[first] : PART == OUTPUTS;
  const int N = p.N, P = p.P;
  const int grp = h / (p.H / p.G);
  const int pc = pb0 + wave * 16 + lc;       // this lane's value channel
  const bool live = pc < P;
  float* sp = p.state + ((long)slot * p.H + h) * N * P;
  const long NP_ = (long)N * P, stride = p.H * NP_;  // of a head, of a run
  float odd = 0.f;                           // NaN behind a value that is not finite
  sc_f32x4 S[NT];                            // rows 16 t + 4 g + r, column pc
  auto each = [&](auto f) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int nn = t * 16 + g * 4 + r;
        if (live && nn < N) S[t][r] = f(S[t][r], (long)nn * P + pc);
      }
  };
#pragma unroll
  for (int t = 0; t < NT; ++t) S[t] = sc_f32x4{0.f, 0.f, 0.f, 0.f};
  if (PART == OUTPUTS && run > run0) {
    const float* at = p.ends + (long)run0 * stride + h * NP_;
    each([&](float, long i) { return at[i]; });
    for (int j = run0 + 1; j < run; ++j) {
      const float fall = p.falls[(long)j * p.H + h];
      at += stride;
      // what is not finite outlives every decay
      each([&](float x, long i) {
        return (fall == 0.f && !(fabsf(x) < INFINITY) ? x : x * fall) + at[i];
      });
    }
    each([&](float x, long) { odd += x * 0.f; return x; });
  } else if (hist > 0) {
    const float* from = PART == OUTPUTS && !ends
                            ? p.scratch + (long)run * stride + h * NP_ : sp;
    each([&](float, long i) { return from[i]; });
    if constexpr (EXACT) each([&](float x, long) { odd += x * 0.f; return x; });
    if constexpr (PART == ENDS) {            // the last run writes the slot
      float* to = p.scratch + (long)run * stride + h * NP_;
      each([&](float x, long i) { return to[i] = x; });
    }
  }
  const float skip = p.skip != nullptr ? p.skip[h] : 0.f;
  const float a_rate = dt_src != nullptr ? expf(p.a_log[h]) : 0.f;
  const float dtb = dt_src != nullptr ? p.dt_bias[h] : 0.f;
  const float a_const = dt_src == nullptr ? p.decay[h] : 0.f;
  const bool neg = a_const < 0.f;            // (-1)^(t - s) beside |a|^(t - s)
  // far enough down that e^it is 0 in fp32, and still exact in the sums; a
  // NaN stays one
  auto low = [](float v) { return v < -1e4f ? -1e4f : v; };
  const float log_const = low(logf(fabsf(a_const)));
  const u16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};

  u16x8 kreg[KU], qreg[KU], vreg;
  float dreg = 0.f;
  auto fetch = [&](int c0) {
    const int rows = min(C, n - c0);
    if constexpr (EXACT) {
      // rows behind the last one and columns of no row come as zeros
      const unsigned ld2 = (unsigned)p.ld_src * 2u;
      const unsigned short* at = src + (long)(first + c0) * p.ld_src;
      auto rsrc = [&](const unsigned short* from, int width) {
        return __builtin_amdgcn_make_buffer_rsrc(
            (void*)from, 0, (unsigned)(rows - 1) * ld2 + (unsigned)width * 2u,
            0x00020000);
      };
      const auto rk = rsrc(at + p.col_b + grp * N, N);
      const auto rq = rsrc(at + p.col_c + grp * N, N);
      const auto rv = rsrc(at + p.col_x + h * P, P);
      auto load8 = [&](const __amdgpu_buffer_rsrc_t& rs, int r, int e, int width) {
        return __builtin_bit_cast(
            u16x8, __builtin_amdgcn_raw_buffer_load_b128(
                       rs, e < width ? (unsigned)r * ld2 + (unsigned)e * 2u : 0xffffff00u,
                       0, 0));
      };
#pragma unroll
      for (int u = 0; u < KU; ++u) {
        const int i = tid + u * 256, r = i / (NP / 8), e = i % (NP / 8) * 8;
        kreg[u] = load8(rk, r, e, N);
        if constexpr (PART != ENDS) qreg[u] = load8(rq, r, e, N);
      }
      vreg = load8(rv, tid / (PB / 8), pb0 + tid % (PB / 8) * 8, P);
      return;
    }
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int i = tid + u * 256, r = i / (NP / 8), e = i % (NP / 8) * 8;
      kreg[u] = zero8;
      qreg[u] = zero8;
      if (r < rows && e < N) {
        const unsigned short* rp = src + (long)(first + c0 + r) * p.ld_src;
        kreg[u] = *reinterpret_cast<const u16x8*>(rp + p.col_b + grp * N + e);
        if constexpr (PART != ENDS)
          qreg[u] = *reinterpret_cast<const u16x8*>(rp + p.col_c + grp * N + e);
      }
    }
    const int r = tid / (PB / 8), e = tid % (PB / 8) * 8;
    vreg = zero8;
    if (r < rows && pb0 + e < P)
      vreg = *reinterpret_cast<const u16x8*>(
          src + (long)(first + c0 + r) * p.ld_src + p.col_x + h * P + pb0 + e);
    if (dt_src != nullptr && tid < rows)
      dreg = bf2f(dt_src[(long)(first + c0 + tid) * p.ld_dt + p.col_dt + h]);
  };
  auto put8 = [&](float* to, const u16x8 from) {
    float f[8];
    bf8_to_f32(from, f);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (p.act) f[i] = silu_f(f[i]);
    *reinterpret_cast<sc_f32x4*>(to) = sc_f32x4{f[0], f[1], f[2], f[3]};
    *reinterpret_cast<sc_f32x4*>(to + 4) = sc_f32x4{f[4], f[5], f[6], f[7]};
  };
  auto mm = [](float a, float b, sc_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  };

  // Eight neighbours of state rows, e .. e + 7. Of 32 rows a lane group takes 4 g ..
  // 4 g + 3 and 16 further on, as the state's accumulators hold them: those lie
  // together.
  auto put_bf = [&](unsigned short* row, int e, const u16x8 from) {
    const u32x4 w = __builtin_bit_cast(u32x4, from);
    unsigned short* at = row + (e & ~31) + (e & 8) * 2 + (e & 16) / 4;
    *reinterpret_cast<sc_u32x2*>(at) = sc_u32x2{w[0], w[1]};
    *reinterpret_cast<sc_u32x2*>(at + 8) = sc_u32x2{w[2], w[3]};
  };

  // Decays and weights of the rows from c0 on, a row a thread, chunks of 32 apart.
  auto scalars = [&](int c0) {
    const int rows = n - c0, row = tid & (C - 1), chunk = EXACT ? tid / C : 0;
    // rows behind the last one: decay 1, weight 0
    float la = 0.f, b = 0.f;
    if (tid < rows) {
      if (dt_src != nullptr) {
        b = softplus_f(dreg + dtb);
        la = low(-a_rate * b);
      } else {
        b = 1.f;
        la = log_const;
      }
    }
    double c = la;
#pragma unroll
    for (int m = 1; m < C; m <<= 1) {
      const double o = __shfl_up(c, m, 32);
      if (row >= m) c += o;
    }
    const double all = __shfl(c, C - 1, 32);
    if (EXACT && chunk >= SB) return;
    const int in = min(C, rows - chunk * C), last = in - 1;
    // EXACT takes powers of two of the differences
    cs2[chunk][row] = EXACT ? c * 1.4426950408889634 : c;
    if (EXACT && row == C - 1)
      fell[chunk] = expf((float)c) * (neg && (in & 1) ? -1.f : 1.f);
    scal[chunk][0][row] = b;
    scal[chunk][1][row] = expf((float)c) * (neg && !(row & 1) ? -1.f : 1.f);
    scal[chunk][2][row] = b * expf((float)(all - c)) *
                          (neg && ((last - row) & 1) ? -1.f : 1.f);
  };
  auto fetch_dt = [&](int c0) {              // EXACT: for the next SB chunks
    if (dt_src != nullptr && tid < SB * C && c0 + tid < n)
      dreg = bf2f(dt_src[(long)(first + c0 + tid) * p.ld_dt + p.col_dt + h]);
  };

  float fall = 1.f;
  fetch(0);
  if constexpr (EXACT) fetch_dt(0);
  for (int c0 = 0; c0 < n; c0 += C) {
    const int rows = min(C, n - c0);
    const int buf = EXACT ? (c0 / C) & 1 : 0, at = c0 / C % SB;
    if constexpr (EXACT) {
      if (at == 0) {
        if (c0 > 0) __syncthreads();         // the last of the SB before is read
        scalars(c0);
        fetch_dt(c0 + SB * C);
        if constexpr (PART != ENDS) {
          __syncthreads();
          const int tr = tid >> 4, sr = tid & 15;
#pragma unroll 1
          for (int b = 0; b < SB; ++b)
#pragma unroll
            for (int i = 0; i < 3; ++i) {    // 16 x 16 on and below the diagonal
              const int t = (i > 0) * 16 + tr, sc = (i > 1) * 16 + sr;
              const bool behind = i == 1 || sr <= tr;
              float x = scal[b][0][sc] *
                        __builtin_amdgcn_exp2f(
                            behind ? (float)(cs2[b][t] - cs2[b][sc]) : 0.f);
              if (neg && ((t - sc) & 1)) x = -x;
              es[b][t][sc] = behind ? x : 0.f;
            }
        }
      }
      el = scal[at][1];
      wl = scal[at][2];
#pragma unroll
      for (int u = 0; u < KU; ++u) {
        const int i = tid + u * 256, r = i / (NP / 8), e = i % (NP / 8) * 8;
        put_bf(kh[buf][r], e, kreg[u]);
        if constexpr (PART != ENDS) put_bf(qh[buf][r], e, qreg[u]);
      }
      *reinterpret_cast<u16x8*>(&vh[buf][tid / (PB / 8)][tid % (PB / 8) * 8]) = vreg;
    } else {
#pragma unroll
    for (int u = 0; u < KU; ++u) {
      const int i = tid + u * 256, r = i / (NP / 8), e = i % (NP / 8) * 8;
      put8(&ks[r][e], kreg[u]);
      if constexpr (PART != ENDS) put8(&qs[r][e], qreg[u]);
    }
    put8(&vs[tid / (PB / 8)][tid % (PB / 8) * 8], vreg);
    }
    if (!EXACT && tid < C) scalars(c0);
    __syncthreads();
    if (c0 + C < n) fetch(c0 + C);

    if constexpr (EXACT) {
      // rows 4 g + j and 16 + 4 g + j of this lane's value channel
      const unsigned short* vp = &vh[buf][g * 4 + (lc >> 2)][wave * 16 + (lc & 3) * 4];
      const sc_u32x2 v0 = read_down(vp), v1 = read_down(vp + 16 * WS);
      const u32x4 vb{v0[0], v0[1], v1[0], v1[1]};
      float vf[8];
      bf8_to_f32(__builtin_bit_cast(u16x8, vb), vf);
      if constexpr (PART != ENDS) {
        u32x4 qf[2][NT / 2];
        sc_f32x4 o[2], o2[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          o[t] = o2[t] = sc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb = 0; kb < NT / 2; ++kb)
            qf[t][kb] = *reinterpret_cast<const u32x4*>(
                &qh[buf][t * 16 + lc][kb * 32 + g * 8]);
        }
        // scores, transposed: row s = 4 g + r, column t = lc; weighted they are the
        // operand of the product with v as they lie
        float w[2][8];
#pragma unroll
        for (int si = 0; si < 2; ++si) {
          sc_f32x4 a[2];
#pragma unroll
          for (int t = 0; t < 2; ++t) a[t] = sc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb = 0; kb < NT / 2; ++kb) {
            const u32x4 kf = *reinterpret_cast<const u32x4*>(
                &kh[buf][si * 16 + lc][kb * 32 + g * 8]);
#pragma unroll
            for (int t = si; t < 2; ++t) a[t] = mm_bf(kf, qf[t][kb], a[t]);
          }
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            if (si > t) {
#pragma unroll
              for (int r = 0; r < 4; ++r) w[t][si * 4 + r] = 0.f;
              continue;
            }
            const sc_f32x4 e4 = *reinterpret_cast<const sc_f32x4*>(
                &es[at][t * 16 + lc][si * 16 + g * 4]);
#pragma unroll
            for (int r = 0; r < 4; ++r) w[t][si * 4 + r] = a[t][r] * e4[r];
          }
        }
        // what the state brings
#pragma unroll
        for (int kb = 0; kb < NT / 2; ++kb) {
          float x[8];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            x[r] = S[2 * kb][r];
            x[4 + r] = S[2 * kb + 1][r];
          }
          const Split8 sp8 = split8<false>(x);
          // two chains a tile: the large parts and the small ones
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            o[t] = mm_bf(qf[t][kb], sp8.part[0], o[t]);
            o2[t] = mm_bf(qf[t][kb], sp8.part[1],
                          mm_bf(qf[t][kb], sp8.part[2], o2[t]));
          }
        }
        const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(
            y + (long)(first + c0) * p.H * P + h * P, 0,
            ((unsigned)(rows - 1) * (unsigned)p.H + 1u) * (unsigned)P * 4u, 0x00020000);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            o[t][r] = (o[t][r] + o2[t][r]) * el[t * 16 + g * 4 + r];
          // and the chunk's own rows
          o[t] = mm_split(split8<true>(w[t]), vb, o[t]);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            odd += o[t][r] * 0.f;
            // rows behind the last and channels of no head are not stored
            const unsigned off =
                ((unsigned)(t * 16 + g * 4 + r) * (unsigned)p.H * (unsigned)P +
                 (unsigned)pc) * 4u;
            __builtin_amdgcn_raw_buffer_store_b32(
                __builtin_bit_cast(unsigned, o[t][r] + skip * vf[t * 4 + r]), ry,
                live ? off : 0xffffff00u, 0, 0);
          }
        }
      }
      // the state behind the chunk
      const float down = fell[at];
      if constexpr (PART == ENDS) fall *= down;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[t][r] *= down;
#pragma unroll
      for (int j = 0; j < 8; ++j) vf[j] *= wl[(j >> 2) * 16 + g * 4 + (j & 3)];
      const Split8 bv = split8<true>(vf);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const unsigned short* kp =
            &kh[buf][g * 4 + (lc >> 2)][t / 2 * 32 + (lc & 3) * 8 + (t & 1) * 4];
        const sc_u32x2 k0 = read_down(kp), k1 = read_down(kp + 16 * HS);
        S[t] = mm_split(u32x4{k0[0], k0[1], k1[0], k1[1]}, bv, S[t]);
      }
      continue;
    }
    sc_f32x4 o[2];
    if constexpr (PART != ENDS) {
    // scores of 16 x 16 rows a wave, weighted
    const int ti = wave >> 1, si = wave & 1;
    if (si <= ti) {
      sc_f32x4 a{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < NT; ++kb) {
        const sc_f32x4 q4 = *reinterpret_cast<const sc_f32x4*>(
            &qs[ti * 16 + lc][kb * 16 + g * 4]);
        const sc_f32x4 k4 = *reinterpret_cast<const sc_f32x4*>(
            &ks[si * 16 + lc][kb * 16 + g * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) a = mm(q4[j], k4[j], a);
      }
      const int sr = si * 16 + lc;
      const double c_s = cs[sr];
      const float b_s = bl[sr];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tr = ti * 16 + g * 4 + r;
        float w = 0.f;
        if (sr <= tr) {
          w = a[r] * expf((float)(cs[tr] - c_s)) * b_s;
          if (neg && ((tr - sr) & 1)) w = -w;
        }
        as[tr][sr] = w;
      }
    }
    // what the state brings
#pragma unroll
    for (int t = 0; t < 2; ++t) o[t] = sc_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < NT; ++kb) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const sc_f32x4 q4 = *reinterpret_cast<const sc_f32x4*>(
            &qs[t * 16 + lc][kb * 16 + g * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[t] = mm(q4[j], S[kb][j], o[t]);
      }
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[t][r] *= el[t * 16 + g * 4 + r];
    __syncthreads();
    }
    // what the chunk's own rows bring
    float vv[2][4];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) vv[b][j] = vs[b * 16 + g * 4 + j][wave * 16 + lc];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) odd += vv[b][j] * 0.f;
    if constexpr (PART != ENDS) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int b = 0; b <= t; ++b) {
        const sc_f32x4 a4 = *reinterpret_cast<const sc_f32x4*>(
            &as[t * 16 + lc][b * 16 + g * 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[t] = mm(a4[j], vv[b][j], o[t]);
      }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tr = t * 16 + g * 4 + r;
        if (tr < rows && live)
          y[(long)(first + c0 + tr) * p.H * P + h * P + pc] =
              o[t][r] + skip * vs[tr][wave * 16 + lc];
      }
    }
    // the state behind the chunk
    const float down = expf((float)cs[C - 1]) *
                       (neg && (rows & 1) ? -1.f : 1.f);
    if constexpr (PART == ENDS) fall *= down;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[t][r] *= down;
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int sr = b * 16 + g * 4 + j;
        const float bv = vv[b][j] * wl[sr];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          S[t] = mm(ks[sr][t * 16 + lc], bv, S[t]);
      }
    __syncthreads();
  }
  // Of EXACT what is not finite, and splits into NaN, shows in the rows (q, k) or in
  // the state (k, v), which keeps it.
  if constexpr (EXACT)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) odd += S[t][r] * 0.f;
  float* own = PART == WHOLE || (PART == OUTPUTS && ends)
                   ? sp
                   : (PART == ENDS ? p.ends : p.scratch) + (long)run * stride +
                         h * NP_;
  if constexpr (PART == ENDS)
    if (tid == 0 && pb0 == 0) p.falls[(long)run * p.H + h] = fall;
  // A value that is infinite or NaN belongs to its own row and those behind
  // it, but the weights of 0 above the diagonal carried it to the rows in
  // front: such columns are walked again row by row, on the state in memory
  // (the slot, or the own place of a run that is not its sequence's last).
  if (__any(odd != 0.f)) {
    auto load = [&](const unsigned short* at) {
      const float f = bf2f(*at);
      return p.act ? silu_f(f) : f;
    };
    if (PART != WHOLE && hist > 0)
#pragma unroll 1
      for (int nn = g; nn < N && live; nn += 4) {
        const long i = (long)nn * P + pc;
        if (run == run0) {                   // of OUTPUTS it is there already
          if (PART == ENDS) own[i] = sp[i];
          continue;
        }
        const float* at = p.ends + (long)run0 * stride + h * NP_ + i;
        float x = *at;
        for (int j = run0 + 1; j < run; ++j) {
          const float f = p.falls[(long)j * p.H + h];
          at += stride;
          x = (f == 0.f && !(fabsf(x) < INFINITY) ? x : x * f) + *at;
        }
        own[i] = x;
      }
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
      const unsigned short* rp = src + (long)(first + i) * p.ld_src;
      float a = a_const, b = 1.f, part = 0.f;
      if (dt_src != nullptr) {
        b = softplus_f(bf2f(dt_src[(long)(first + i) * p.ld_dt + p.col_dt + h])
                       + dtb);
        a = expf(-a_rate * b);
      }
      const float v = live ? load(rp + p.col_x + h * P + pc) : 0.f;
#pragma unroll 1
      for (int nn = g; nn < N && live; nn += 4) {
        float* at = own + (long)nn * P + pc;
        const float old = i > 0 || hist > 0 ? *at : 0.f;
        *at = a * old + b * load(rp + p.col_b + grp * N + nn) * v;
        if constexpr (PART != ENDS)
          part += *at * load(rp + p.col_c + grp * N + nn);
      }
      if constexpr (PART != ENDS) {
        part += __shfl_xor(part, 16, 64);
        part += __shfl_xor(part, 32, 64);
        if (g == 0 && live)
          y[(long)(first + i) * p.H * P + h * P + pc] = part + skip * v;
      }
    }
    return;
  }
  if (PART == ENDS || ends) each([&](float x, long i) { return own[i] = x; });
}

// Single rows (decode): the state itself is the traffic, so one workgroup
// per (sequence, head) streams it once with 16-byte accesses — a lane
// owns 4 neighbouring value channels of every RP-th state row — updates it
// in place and reduces y over the rows through LDS. More rows of a
// sequence, should a batch bring them, are walked one after the other.
// U state rows of a lane are in flight, the first of them beside the token's
// values; 0: each behind the store of the one before, as the compiler places it
// (step_flight).
template <typename TS, int U>
__global__ __launch_bounds__(256) void state_step_kernel(
    float* __restrict__ y, const TS* __restrict__ src,
    const TS* __restrict__ dt_src, ScanArgs p) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int N = p.N, P = p.P, P4 = P / 4, RP = 256 / P4;
  float* vs = sm;                 // [P]      (16-byte reads: P % 4 == 0)
  float* part = vs + P;           // [RP][P]
  float* ks = part + RP * P;      // [N]
  float* qs = ks + N;             // [N]
  __shared__ float ab[2];
  const int s = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x;
  const int cg = tid % P4, r0 = tid / P4;
  const int first = p.seq_first[s], n = p.seq_rows[s];
  if (first < 0 || n < 1 || first + n > p.T) return;
  const int slot = min(max(p.state_slots[s], 0), p.nslots - 1);
  const int hist = p.pos32[first];
  const int g = h / (p.H / p.G);
  float* sp = p.state + ((long)slot * p.H + h) * N * P;
  const float skip = p.skip != nullptr ? p.skip[h] : 0.f;
  f32x4 S[U > 0 ? U : 1];
  auto bring = [&](int n0, bool fresh) {
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const int nn = n0 + j * RP;
      S[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (!fresh && r0 < RP && nn < N)
        S[j] = *reinterpret_cast<const f32x4*>(sp + (long)nn * P + cg * 4);
    }
  };
  if constexpr (U > 0) bring(r0, hist <= 0);
  for (int r = 0; r < n; ++r) {
    const TS* rp = src + (long)(first + r) * p.ld_src;
    __syncthreads();
    for (int i = tid; i < N; i += 256) {
      float kv = ld(rp + p.col_b + g * N + i), qv = ld(rp + p.col_c + g * N + i);
      if (p.act) { kv = silu_f(kv); qv = silu_f(qv); }
      ks[i] = kv;
      qs[i] = qv;
    }
    for (int i = tid; i < P; i += 256) {
      float v = ld(rp + p.col_x + h * P + i);
      vs[i] = p.act ? silu_f(v) : v;
    }
    if (tid == 0) {
      if (dt_src != nullptr) {
        const float dt = softplus_f(
            ld(dt_src + (long)(first + r) * p.ld_dt + p.col_dt + h) + p.dt_bias[h]);
        ab[0] = expf(-expf(p.a_log[h]) * dt);
        ab[1] = dt;
      } else {
        ab[0] = p.decay[h];
        ab[1] = 1.f;
      }
    }
    __syncthreads();
    const float a = ab[0], b = ab[1];
    const bool fresh = hist <= 0 && r == 0;      // start from a zero state
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (r0 < RP) {
      const f32x4 v4 = *reinterpret_cast<const f32x4*>(vs + cg * 4);
      auto put = [&](f32x4 state, int nn) {
        const float bk = b * ks[nn], qn = qs[nn];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          state[k] = a * state[k] + bk * v4[k];
          acc[k] += state[k] * qn;
        }
        *reinterpret_cast<f32x4*>(sp + (long)nn * P + cg * 4) = state;
      };
      if constexpr (U == 0) {
        for (int nn = r0; nn < N; nn += RP)
          put(fresh ? f32x4{0.f, 0.f, 0.f, 0.f}
                    : *reinterpret_cast<const f32x4*>(sp + (long)nn * P + cg * 4), nn);
      } else {
        for (int n0 = r0; n0 < N; n0 += U * RP) {
          if (n0 > r0 || r > 0) bring(n0, fresh);
#pragma unroll
          for (int j = 0; j < U; ++j) {
            const int nn = n0 + j * RP;
            if (nn >= N) break;
            put(S[j], nn);
          }
        }
      }
      *reinterpret_cast<f32x4*>(part + r0 * P + cg * 4) = acc;
    }
    __syncthreads();
    for (int i = tid; i < P; i += 256) {
      float o = skip * vs[i];
      for (int k = 0; k < RP; ++k) o += part[k * P + i];
      y[(long)(first + r) * p.H * P + h * P + i] = o;
    }
  }
}

// State rows of a lane in flight, by the rows that it has and the workgroups. Few
// workgroups wait for their own rows, with many each memory channel has work anyway, and
// a state's few rows then only come to it in another order. us, one by one / four /
// eight (less than 3 % is within the runs):
//   2 rows:  256 workgroups 5.0 / 4.9 / 5.1, 1024 7.2 / 6.8 / 7.0, 2048 12.7 / 10.8 / 11.9,
//            4096 20.0 / 20.9 / 22.8, 8192 33.5 / 34.3 / 38.5
//   4:       512 7.0 / 6.5 / 6.6, 1024 12.7 / 9.8 / 10.0, 2048 18.6 / 19.7 / 19.8, 4096
//            31.0 / 32.3 / 33.5, 8192 56.5 / 58.2 / 59.6
//   8:       256 7.6 / 7.0 / 6.8, 512 13.4 / 10.2 / 10.0, 1024 18.6 / 19.2 / 18.5, 2048
//            30.8 / 30.5 / 32.5, 4096 58.9 / 55.1 / 56.9, 8192 105.8 / 106.2 / 108.1
//   16:      256 16.5 / 12.8 / 9.7, 1024 37.3 / 37.4 / 36.0, 2048 65.6 / 60.3 / 60.6,
//            4096 121.6 / 113.1 / 112.5, 8192 217.6 / 217.5 / 218.1
int step_flight(int N, int P, long workgroups) {
  const int rows = (N + 1024 / P - 1) / (1024 / P);
  if (rows > 8) return 8;
  if (rows > 4) return workgroups <= 1024 ? 8 : 4;
  return workgroups <= 1024 ? 4 : 0;
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

// grid (T, groups): one workgroup per (row, part). gate_first 1: u = y *
// silu(gate), out = u / rms(u) * w; 0: out = y / rms(y) * w * sigmoid(gate);
// 2: out = y / rms(y) * w * silu(gate). ysc [T, groups] (or null) multiplies y
// first.
template <typename TG, typename TO>
__global__ __launch_bounds__(ROW_THREADS) void gated_group_norm_kernel(
    TO* __restrict__ out, const float* __restrict__ y,
    const float* __restrict__ ysc, const TG* __restrict__ gate, long ld_gate, const float* __restrict__ w,
    int C, int gs, float eps, int gate_first) {
  __shared__ float red[4];
  const long t = blockIdx.x;
  const int c0 = blockIdx.y * gs;
  const float* yr = y + t * C + c0;
  const TG* gr = gate + t * ld_gate + c0;
  const float sc = ysc != nullptr ? ysc[t * gridDim.y + blockIdx.y] : 1.f;
  float ss = 0.f;
  for (int i = threadIdx.x; i < gs; i += ROW_THREADS) {
    float u = yr[i] * sc;
    if (gate_first == 1) u *= silu_f(ld(gr + i));
    ss += u * u;
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
  for (int i = threadIdx.x; i < gs; i += ROW_THREADS) {
    const float gv = ld(gr + i);
    float u = yr[i] * sc;
    if (gate_first == 1) u = u * silu_f(gv) * inv * w[c0 + i];
    else if (gate_first == 2) u = u * inv * w[c0 + i] * silu_f(gv);
    else u = u * inv * w[c0 + i] * sigmoid_f(gv);
    st(out + t * C + c0 + i, u);
  }
}

// The same for bf16 gates and outputs with parts of a multiple of 4 and at
// most 4096 channels: a lane keeps its 4 x NV channels in registers between
// the sum of squares and the store (one pass over y and the gate).
template <int NV>
__global__ __launch_bounds__(ROW_THREADS) void gated_group_norm_vec_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ y,
    const float* __restrict__ ysc, const unsigned short* __restrict__ gate, long ld_gate,
    const float* __restrict__ w, int C, int gs, float eps, int gate_first) {
  __shared__ float red[4];
  const long t = blockIdx.x;
  const int c0 = blockIdx.y * gs;
  const float* yr = y + t * C + c0;
  const unsigned short* gr = gate + t * ld_gate + c0;
  const float sc = ysc != nullptr ? ysc[t * gridDim.y + blockIdx.y] : 1.f;
  float u[NV][4], gv[NV][4];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (threadIdx.x + j * ROW_THREADS) * 4;
    if (i < gs) {
      const f32x4 yv = *reinterpret_cast<const f32x4*>(yr + i);
      const u16x4 g4 = *reinterpret_cast<const u16x4*>(gr + i);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        gv[j][k] = bf2f(g4[k]);
        u[j][k] = yv[k] * sc;
        if (gate_first == 1) u[j][k] *= silu_f(gv[j][k]);
        ss += u[j][k] * u[j][k];
      }
    }
  }
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (threadIdx.x + j * ROW_THREADS) * 4;
    if (i < gs) {
      const f32x4 wv = *reinterpret_cast<const f32x4*>(w + c0 + i);
      u16x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float r = u[j][k] * inv * wv[k];
        if (gate_first == 0) r *= sigmoid_f(gv[j][k]);
        else if (gate_first == 2) r *= silu_f(gv[j][k]);
        o[k] = f2bf(r);
      }
      *reinterpret_cast<u16x4*>(out + t * C + c0 + i) = o;
    }
  }
}

// Parts of more than 256 and up to 512 NV channels, a multiple of 8, of rows at 16-byte
// addresses: a wave to a part, without the LDS or a barrier. Bound by the rows' bytes:
// 7032 rows of 8 parts of 512 47.6 us (a workgroup to a part, half of whose lanes had
// no channels, with expf and a division 68.6).
template <int NV>
__global__ __launch_bounds__(ROW_THREADS) void gated_group_norm_wave_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ y,
    const float* __restrict__ ysc, const unsigned short* __restrict__ gate, long ld_gate,
    const float* __restrict__ w, long units, int groups, int gs, float eps,
    int gate_first) {
  const long unit = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (unit >= units) return;
  const long t = unit / groups;
  const int grp = (int)(unit % groups), c0 = grp * gs, lane = threadIdx.x & 63;
  const float* yr = y + unit * gs;
  const unsigned short* gr = gate + t * ld_gate + c0;
  const float sc = ysc != nullptr ? ysc[unit] : 1.f;
  f32x4 yv[NV][2], wv[NV][2];
  u16x8 g8[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (lane + j * 64) * 8;
    if (i >= gs) break;
    g8[j] = *reinterpret_cast<const u16x8*>(gr + i);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      yv[j][k] = *reinterpret_cast<const f32x4*>(yr + i + k * 4);
      wv[j][k] = *reinterpret_cast<const f32x4*>(w + c0 + i + k * 4);
    }
  }
  float u[NV][8], ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if ((lane + j * 64) * 8 >= gs) break;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      u[j][k] = yv[j][k / 4][k % 4] * sc;
      if (gate_first == 1) u[j][k] *= silu_f(bf2f(g8[j][k]));
      ss += u[j][k] * u[j][k];
    }
  }
  ss = wave_reduce_sum(ss);
  const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (lane + j * 64) * 8;
    if (i >= gs) break;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      u[j][k] = u[j][k] * inv * wv[j][k / 4][k % 4];
      if (gate_first == 0) u[j][k] *= sigmoid_f(bf2f(g8[j][k]));
      else if (gate_first == 2) u[j][k] *= silu_f(bf2f(g8[j][k]));
    }
    *reinterpret_cast<u16x8*>(out + unit * gs + i) = f32_to_bf8(u[j]);
  }
}

// bf16 gates and outputs, parts of a multiple of 4 and at most 256
// channels (per-head norms): LPG lanes share a part, 4 channels each in one
// step, a wave takes 64 / LPG parts of a row and a workgroup four times that.
template <int LPG>
__global__ __launch_bounds__(ROW_THREADS) void gated_group_norm_small_kernel(
    unsigned short* __restrict__ out, const float* __restrict__ y,
    const float* __restrict__ ysc, const unsigned short* __restrict__ gate, long ld_gate,
    const float* __restrict__ w, int C, int gs, int groups, float eps,
    int gate_first) {
  constexpr int GPW = 64 / LPG;
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int grp = (blockIdx.y * 4 + wave) * GPW + lane / LPG;
  const int c = (lane % LPG) * 4;
  const bool live = grp < groups && c < gs;
  const int c0 = grp * gs + c;
  float u[4] = {0.f, 0.f, 0.f, 0.f}, gv[4] = {0.f, 0.f, 0.f, 0.f};
  float ss = 0.f;
  if (live) {
    const f32x4 yv = *reinterpret_cast<const f32x4*>(y + t * C + c0);
    const u16x4 g4 = *reinterpret_cast<const u16x4*>(gate + t * ld_gate + c0);
    const float sc = ysc != nullptr ? ysc[t * groups + grp] : 1.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      gv[k] = bf2f(g4[k]);
      u[k] = yv[k] * sc;
      if (gate_first == 1) u[k] *= silu_f(gv[k]);
      ss += u[k] * u[k];
    }
  }
#pragma unroll
  for (int m = LPG / 2; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, WAVE_SIZE);
  if (!live) return;
  const float inv = 1.0f / sqrtf(ss / (float)gs + eps);
  const f32x4 wv = *reinterpret_cast<const f32x4*>(w + c0);
  u16x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float r = u[k] * inv * wv[k];
    if (gate_first == 0) r *= sigmoid_f(gv[k]);
    else if (gate_first == 2) r *= silu_f(gv[k]);
    o[k] = f2bf(r);
  }
  *reinterpret_cast<u16x4*>(out + t * C + c0) = o;
}

template <typename TS, typename TD, int NR, int TPP>
void scan_launch(float* y, const void* src, const void* dt, const ScanArgs& p,
                 int nseq, hipStream_t s) {
  constexpr int PL = 64 / TPP;
  dim3 grid(nseq, p.H, (p.P + PL - 1) / PL);
  state_scan_kernel<TS, TD, NR, TPP, (NR * TPP > 256 ? 8 : 16)>
      <<<grid, 64, 0, s>>>(y, (const TS*)src, (const TD*)dt, p);
}

// Rows of the state per lane (NR) and lanes per value channel (TPP): the
// fewest lanes per channel that keep NR <= 32, but no more channels per wave
// than the head has.
constexpr int CHUNK_ROWS = 24;

// 16-byte staging: bf16 rows whose sizes and columns are multiples of 8
bool vec_rows(int N, int P, long ld_src, int col_x, int col_b, int col_c) {
  return N % 8 == 0 && P % 8 == 0 && ld_src % 8 == 0 && col_x % 8 == 0 &&
         col_b % 8 == 0 && col_c % 8 == 0;
}

// Chunks on the matrix instructions from CHUNK_ROWS rows a sequence on (on
// average: the sizes themselves are on the device), where a wave's 16 value
// channels and 16-row state tiles are not mostly padding
bool chunk_rows(int bf, bool vec, int N, int P, long T, int nseq) {
  return bf && vec && N >= 32 && N <= 128 && P >= 32 &&
         T >= (long)CHUNK_ROWS * nseq;
}

// batches of single rows: the streaming step kernel, when the value size splits
// a workgroup evenly into 16-byte columns
bool step_rows(int single, int N, int P) {
  const int P4 = P / 4;
  return single && P % 4 == 0 && P4 >= 1 && P4 <= 256 && 256 % P4 == 0 &&
         (size_t)(2 * N + P + (256 / P4) * P) * sizeof(float) <= 48 * 1024;
}

template <typename TS, typename TD>
bool scan_pick(float* y, const void* src, const void* dt, const ScanArgs& p,
               int nseq, hipStream_t s) {
  int tpp = 1;
  while (tpp < 8 && ((p.N + tpp - 1) / tpp > 32 || 64 / tpp > max(p.P, 8)))
    tpp *= 2;
  const bool vec = vec_rows(p.N, p.P, p.ld_src, p.col_x, p.col_b, p.col_c);
  if (chunk_rows(sizeof(TS) == 2, vec, p.N, p.P, p.T, nseq)) {
#define CHUNKS_AS(NT, PART, GROUPS, EXACT)                                   \
  state_chunk_kernel<NT, PART, EXACT>                                        \
      <<<dim3(GROUPS, p.H, (p.P + 63) / 64), 256, 0, s>>>(                   \
          y, (const unsigned short*)src, (const unsigned short*)dt, p)
#define CHUNKS(NT, PART, GROUPS)                                             \
  if (p.act) CHUNKS_AS(NT, PART, GROUPS, false);                             \
  else CHUNKS_AS(NT, PART, GROUPS, true)
#define CHUNKS_NT(NT)                                                        \
  if (p.ncut > 0) {                                                          \
    CHUNKS(NT, ENDS, p.ncut);                                                \
    CHUNKS(NT, OUTPUTS, p.nruns);                                            \
  } else {                                                                   \
    CHUNKS(NT, WHOLE, nseq);                                                 \
  }
    if (p.N <= 64) { CHUNKS_NT(4) } else { CHUNKS_NT(8) }
#undef CHUNKS_NT
#undef CHUNKS
#undef CHUNKS_AS
    return true;
  }
  // few workgroups (long portions of few sequences): more lanes per channel
  // make more, smaller ones, so that every SIMD holds two waves
  while (vec && sizeof(TS) == 2 && tpp < 8 && (p.N + tpp - 1) / tpp >= 16 &&
         (long)nseq * p.H * ((p.P + 4 * (64 / tpp) - 1) / (4 * (64 / tpp))) < 512)
    tpp *= 2;
  const int nr = (p.N + tpp - 1) / tpp;
#define SCAN_CASE(NRV, TPPV)                                              \
  if (tpp == TPPV && nr <= NRV) {                                         \
    constexpr bool fits = sizeof(TS) == 2 &&                              \
        (4 * CH * TPPV * (NRV + 4) + 2 * CH * 4 * (64 / TPPV) + 4 * CH) * 4 \
            <= 60 * 1024;                                                 \
    if constexpr (fits) if (vec) {                                        \
      constexpr int PBV = 4 * (64 / TPPV);                                \
      dim3 grid(nseq, p.H, (p.P + PBV - 1) / PBV);                        \
      state_scan_vec_kernel<NRV, TPPV><<<grid, 256, 0, s>>>(              \
          y, (const unsigned short*)src, (const unsigned short*)dt, p);   \
      return true;                                                        \
    }                                                                     \
    scan_launch<TS, TD, NRV, TPPV>(y, src, dt, p, nseq, s);               \
    return true;                                                          \
  }
#define SCAN_TPP(TPPV) \
  SCAN_CASE(4, TPPV) SCAN_CASE(8, TPPV) SCAN_CASE(16, TPPV) SCAN_CASE(32, TPPV)
  SCAN_TPP(1) SCAN_TPP(2) SCAN_TPP(4) SCAN_TPP(8) SCAN_CASE(64, 8)
#undef SCAN_TPP
#undef SCAN_CASE
  return false;
}

}  // namespace

int state_scan_max_state() { return 8 * 64; }

// Whether a call of these sizes may be cut into runs: the chunk kernel takes it.
bool state_scan_cuts(int src_bf, int single, int N, int P, long ld_src, int col_x,
                     int col_b, int col_c, long T, int nseq) {
  return !step_rows(single, N, P) &&
         chunk_rows(src_bf, vec_rows(N, P, ld_src, col_x, col_b, col_c), N, P, T,
                    nseq);
}

// src_bf: src and dt_src are bf16 (else fp32). single: the caller expects
// one row per sequence (a hint: any batch is still computed correctly).
// runs: the sequences cut into nruns runs of rows, where state_scan_cuts; the
// first ncut of them (0: no runs) with ends and scratch [ncut, H, N, P] and falls
// [ncut, H].
// Returns 0 when no instantiation covers the sizes.
int state_scan_launch(float* y, const void* src, long ld_src, int col_x,
                      int col_b, int col_c, const void* dt_src, long ld_dt,
                      int col_dt, int H, int G, int N, int P, int act,
                      const float* dt_bias, const float* a_log,
                      const float* skip, const float* decay, float* state,
                      const int* seq_first, const int* seq_rows,
                      const int* state_slots, const int* pos32, int nseq,
                      int nslots, int T, int src_bf, int single,
                      const int* runs, int nruns, int ncut, float* ends,
                      float* scratch,
                      float* falls, hipStream_t s) {
  if (T <= 0 || nseq <= 0) return 1;
  ScanArgs p;
  p.runs = runs; p.nruns = nruns; p.nseq = nseq; p.ncut = ncut; p.ends = ends;
  p.scratch = scratch; p.falls = falls;
  p.ld_src = ld_src; p.ld_dt = ld_dt; p.col_x = col_x; p.col_b = col_b;
  p.col_c = col_c; p.col_dt = col_dt; p.H = H; p.G = G; p.N = N; p.P = P;
  p.act = act; p.dt_bias = dt_bias; p.a_log = a_log; p.skip = skip;
  p.decay = decay; p.state = state; p.seq_first = seq_first;
  p.seq_rows = seq_rows; p.state_slots = state_slots; p.pos32 = pos32;
  p.nslots = nslots; p.T = T;
  if (step_rows(single, N, P)) {
    const int P4 = P / 4;
    const size_t smem = (size_t)(2 * N + P + (256 / P4) * P) * sizeof(float);
#define STEP(T_, U)                                                          \
  state_step_kernel<T_, U><<<dim3(nseq, H), 256, smem, s>>>(                  \
      y, (const T_*)src, (const T_*)dt_src, p)
    const int flight = step_flight(N, P, (long)nseq * H);
    if (src_bf && flight == 8) STEP(unsigned short, 8);
    else if (src_bf && flight == 4) STEP(unsigned short, 4);
    else if (src_bf) STEP(unsigned short, 0);
    else if (flight == 8) STEP(float, 8);
    else if (flight == 4) STEP(float, 4);
    else STEP(float, 0);
#undef STEP
    return 1;
  }
  if (src_bf)
    return scan_pick<unsigned short, unsigned short>(y, src, dt_src, p, nseq, s);
  return scan_pick<float, float>(y, src, dt_src, p, nseq, s);
}

void gated_group_norm_launch(void* out, const float* y, const float* ysc,
                             const void* gate,
                             long ld_gate, const float* w, int T, int C,
                             int groups, float eps, int gate_first, int gate_bf,
                             int out_bf, hipStream_t s) {
  if (T <= 0) return;
  dim3 grid(T, groups);
  const int gs = C / groups;
  if (gate_bf && out_bf && gs % 4 == 0 && C % 4 == 0 && ld_gate % 4 == 0 &&
      gs <= 256 && groups > 1 && ((uintptr_t)gate % 8) == 0) {
    int lpg = 1;
    while (lpg * 4 < gs) lpg *= 2;
    const int gpb = 4 * (64 / lpg);
    const dim3 sgrid(T, (groups + gpb - 1) / gpb);
#define GGN(L)                                                               \
  gated_group_norm_small_kernel<L><<<sgrid, ROW_THREADS, 0, s>>>(            \
      (unsigned short*)out, y, ysc, (const unsigned short*)gate, ld_gate, w, C,   \
      gs, groups, eps, gate_first)
    switch (lpg) {
      case 1: GGN(1); break;
      case 2: GGN(2); break;
      case 4: GGN(4); break;
      case 8: GGN(8); break;
      case 16: GGN(16); break;
      case 32: GGN(32); break;
      default: GGN(64); break;
    }
#undef GGN
    return;
  }
  // A wave to a part from 6144 of them on; of fewer a part's own chain is what is left,
  // which a workgroup shares. us, workgroup / wave, gate first and behind, parts of 512:
  // 512 2.9 / 4.1 and 2.8 / 3.5, 2048 4.1 / 5.3 and 4.0 / 4.3, 4096 6.7 / 7.3 and 6.6 / 6.3,
  // 6144 8.7 / 8.9 and 8.4 / 7.5, 24576 27 / 24 and 27 / 19; of 1024 2048 5.9 / 7.2 and 5.8 /
  // 6.4, 6144 11.9 / 12.2 and 11.8 / 11.5; of 264 4096 5.5 / 6.2 and 5.5 / 5.2.
  if (gate_bf && out_bf && gs % 8 == 0 && C == groups * gs && ld_gate % 8 == 0 &&
      gs <= 1024 && groups > 1 && (long)T * groups >= 6144 &&
      (((uintptr_t)gate | (uintptr_t)y | (uintptr_t)w | (uintptr_t)out) % 16) == 0) {
    const long units = (long)T * groups;
    const dim3 wgrid((unsigned)((units + 3) / 4));
    if (gs <= 512)
      gated_group_norm_wave_kernel<1><<<wgrid, ROW_THREADS, 0, s>>>(
          (unsigned short*)out, y, ysc, (const unsigned short*)gate, ld_gate, w,
          units, groups, gs, eps, gate_first);
    else
      gated_group_norm_wave_kernel<2><<<wgrid, ROW_THREADS, 0, s>>>(
          (unsigned short*)out, y, ysc, (const unsigned short*)gate, ld_gate, w,
          units, groups, gs, eps, gate_first);
    return;
  }
  if (gate_bf && out_bf && gs % 4 == 0 && C % 4 == 0 && ld_gate % 4 == 0 &&
      gs <= 4096 && ((uintptr_t)gate % 8) == 0) {
    if (gs <= 1024)
      gated_group_norm_vec_kernel<1><<<grid, ROW_THREADS, 0, s>>>(
          (unsigned short*)out, y, ysc, (const unsigned short*)gate, ld_gate, w, C,
          gs, eps, gate_first);
    else
      gated_group_norm_vec_kernel<4><<<grid, ROW_THREADS, 0, s>>>(
          (unsigned short*)out, y, ysc, (const unsigned short*)gate, ld_gate, w, C,
          gs, eps, gate_first);
    return;
  }
  if (gate_bf) {
    if (out_bf)
      gated_group_norm_kernel<unsigned short, unsigned short>
          <<<grid, ROW_THREADS, 0, s>>>((unsigned short*)out, y, ysc,
                                        (const unsigned short*)gate, ld_gate, w,
                                        C, gs, eps, gate_first);
    else
      gated_group_norm_kernel<unsigned short, float><<<grid, ROW_THREADS, 0, s>>>(
          (float*)out, y, ysc, (const unsigned short*)gate, ld_gate, w, C, gs, eps,
          gate_first);
  } else {
    if (out_bf)
      gated_group_norm_kernel<float, unsigned short><<<grid, ROW_THREADS, 0, s>>>(
          (unsigned short*)out, y, ysc, (const float*)gate, ld_gate, w, C, gs, eps,
          gate_first);
    else
      gated_group_norm_kernel<float, float><<<grid, ROW_THREADS, 0, s>>>(
          (float*)out, y, ysc, (const float*)gate, ld_gate, w, C, gs, eps,
          gate_first);
  }
}
