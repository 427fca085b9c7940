// Torch bindings for the gpustack_amd HIP ops (native ROCm: no hipify,
// streams come straight from c10::hip).
#include <torch/extension.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include "pinned_words.h"

// launchers (defined in the .hip translation units)
void rms_norm_launch(void*, const void*, const void*, const long*, void*, long, float, int, int, hipStream_t);
void fused_add_rms_norm_launch(void*, const void*, void*, const void*, const void*, int, const long*, int, float, int, int, int, hipStream_t);
void rope_neox_launch(const long*, void*, void*, const float*, int, int, int, int, int, long, long, hipStream_t);
void silu_and_mul_launch(void*, const void*, long, int, hipStream_t);
void reshape_and_cache_launch(const void*, const void*, void*, void*, const long*, int, int, int, int, long, long, int, hipStream_t);
void greedy_sample_launch(long*, long*, const void*, int, int, hipStream_t);
void mla_decode_launch(float*, const void*, const void*, const int*, const int*, int, int, int, int, int, int, float, int*, hipStream_t);
void qkv_store_launch(void*, const float*, int, const void*, const void*, const float*, const long*, const long*, void*, void*, long, int, int, int, int, float, int, int*, hipStream_t);
struct DecodeParts { int n, least, heads; };
struct NewRows {
  const unsigned short* rows;
  const float* parts;
  int nparts;
  const unsigned short *q_norm, *k_norm;
  const float* cos_sin;
  const long *positions, *slots;
  float eps;
};
DecodeParts decode_parts(int, int, int, int, int, int, int, int);
void paged_attn_decode_launch(void*, const void*, const void*, const void*, const int*, const int*, float*, DecodeParts, int, int, int, int, int, float, long, int, const float*, int, float, const NewRows*, int*, hipStream_t);
void flash_prefill_launch(void*, const void*, const void*, const void*, const int*, const int*, const int*, int, int, int, int, int, float, long, long, long, const float*, int, float, int*, hipStream_t);
void flash_prefill_paged_launch(void*, const void*, const void*, const void*, const int*, const int*, const int*, const int*, const int*, const int*, int, int, int, int, int, float, long, const float*, int, float, int*, hipStream_t);
void mfma_probe_launch(float*, const void*, const void*, hipStream_t);
void skinny_gemm_launch(void*, const void*, const void*, void*, int, int, int, int, hipStream_t);
void gemm8_launch(void*, const void*, const void*, int, int, int, int, int*, hipStream_t);
void skinny_gemm_v2_launch(void*, const void*, const void*, void*, int, int, int, int, hipStream_t);
void gemm_lab_launch(void*, const void*, const void*, int, int, int, int, int*, hipStream_t);
void moe_tiles_launch(int*, int*, const int*, int, int, hipStream_t);
void moe_down_scale_launch(void*, const void*, const void*, const int*, const int*, const int*, const float*, const void*, const int*, const int*, long, int, int, int, int*, hipStream_t);
void moe_topk_launch(int*, float*, const float*, int, int, int, int, int, int*, hipStream_t);
void moe_choose_launch(int*, float*, int*, int*, int*, int*, int*, int*, const float*, int, int, int, int, int, int*, hipStream_t);
void moe_route_launch(int*, float*, const void*, const void*, int, int, int, int, int, int*, hipStream_t);
int moe_sort_slices(int);
void moe_sort_launch(int*, int*, float*, const float*, int*, int*, int*, int*, int*, const int*, int, int, int, int*, hipStream_t);
bool moe_wide_takes(int, long, long, int, int, int);
void moe_wide_launch(int, void*, const void*, const void*, const int*, const float*, const int*, const int*, long, long, int, int, int, hipStream_t);
void moe_sum_launch(void*, const void*, long, int, int, hipStream_t);
void moe_tile_launch(int, void*, const void*, const void*, const int*, const int*, const int*, const int*, const int*, const float*, const void*, int, long, int, int, int, int*, hipStream_t);
void moe_few_launch(int, void*, const void*, const void*, const int*, const int*, const int*, const int*, const int*, const float*, long, long, int, int, int, int*, hipStream_t);
void rows_tile_launch(void*, void*, const void*, const void*, int, int, int, long, int, int, int, int*, hipStream_t);
void rows_gemm_launch(void*, const void*, const void*, int, int, int, long, int*, hipStream_t);
bool w4_has(int, int);
bool w4_cuts(int, int, int);
bool w4_by_rows(int, int, int);
bool w4_silu_wins(int, int, int);
void wide_launch(int, void*, const void*, const void*, int, int, int, long, int, int, int, int*, hipStream_t);
int w4_splits(int, int, int);
void w4_parts_launch(float*, const void*, const void*, const void*, const void*, int, int, int, int, hipStream_t);
void w4_silu_launch(void*, const void*, const void*, const void*, const void*, int, int, int, hipStream_t);
void w4_tile_launch(void*, const void*, const void*, const void*, const void*, int, int, int, hipStream_t);
void w4_rows_launch(void*, const void*, const void*, const void*, const void*, int, int, int, hipStream_t);
void rows_join_launch(void*, const float*, long, int, hipStream_t);
void w4_dequant_launch(void*, const void*, const void*, const void*, long, int, int*, hipStream_t);

#define HIP_CHECK_LAST()                                                     \
  do {                                                                       \
    hipError_t e_ = hipGetLastError();                                       \
    TORCH_CHECK(e_ == hipSuccess, "HIP kernel launch failed: ",              \
                hipGetErrorString(e_));                                      \
  } while (0)

namespace {

hipStream_t cur_stream(const at::Tensor& t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

void check_bf16(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

void check_i32(const at::Tensor& t, long n, const char* name) {
  TORCH_CHECK(t.is_cuda() && t.scalar_type() == at::kInt && t.is_contiguous()
              && t.numel() >= n, name, " must be a GPU int32 list of ", n);
}

bool is_fp8_cache(const at::Tensor& t) {
  return t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte;
}

void check_cache(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16 || is_fp8_cache(t),
              name, " must be bf16 or fp8-e4m3");
  TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
}

// [T, H, D] tensor allowed a non-contiguous row stride (view into a fused
// qkv buffer); heads and dims must stay contiguous.
long row_stride_3d(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.is_cuda(), name, " must be on GPU");
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bf16");
  TORCH_CHECK(t.dim() == 3, name, " must be [T, H, D]");
  TORCH_CHECK(t.stride(2) == 1 && t.stride(1) == t.size(2),
              name, " heads/dims must be contiguous");
  return t.stride(0);
}

void rms_norm(at::Tensor out, at::Tensor input, at::Tensor weight, double eps) {
  check_bf16(out, "out"); check_bf16(input, "input"); check_bf16(weight, "weight");
  const int H = input.size(-1);
  const long T = input.numel() / H;
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  rms_norm_launch(out.data_ptr(), input.data_ptr(), weight.data_ptr(), nullptr,
                  nullptr, 0, (float)eps, (int)T, H, cur_stream(input));
  HIP_CHECK_LAST();
}

// x = the rows of the tokens, out their norm
void embed_rms_norm(at::Tensor out, at::Tensor x, at::Tensor tokens,
                    at::Tensor embed, at::Tensor weight, double eps) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(embed, "embed");
  check_bf16(weight, "weight");
  const int H = embed.size(1);
  const long T = tokens.numel();
  TORCH_CHECK(tokens.is_cuda() && tokens.scalar_type() == at::kLong &&
              tokens.is_contiguous(), "tokens must be int64 on GPU");
  TORCH_CHECK(H % 8 == 0 && weight.numel() == H && x.numel() == T * H &&
              out.numel() == T * H, "embed_rms_norm shapes");
  if (T == 0) return;
  rms_norm_launch(out.data_ptr(), embed.data_ptr(), weight.data_ptr(),
                  tokens.data_ptr<long>(), x.data_ptr(), embed.size(0),
                  (float)eps, (int)T, H, cur_stream(x));
  HIP_CHECK_LAST();
}

// fp32 parts [n, rows, cols] of a product cut over k, not added up
bool at_16(const at::Tensor& t) { return (uintptr_t)t.data_ptr() % 16 == 0; }

const float* check_parts(const at::Tensor& p, long rows, long cols) {
  TORCH_CHECK(p.is_cuda() && p.scalar_type() == at::kFloat &&
              p.is_contiguous() && p.dim() == 3 && p.size(0) >= 1 &&
              p.size(1) == rows && p.size(2) == cols,
              "parts must be fp32 [n, rows, cols]");
  return p.data_ptr<float>();
}

// what a norm adds to its stream besides rows: fp32 parts [n, rows, cols], or bf16
// rows of a row's experts [rows, n, cols]
struct Addend { const void* data; int chosen, n; };

Addend norm_addend(const at::Tensor& p, long rows, long cols) {
  if (p.scalar_type() == at::kFloat)
    return {check_parts(p, rows, cols), 0, (int)p.size(0)};
  check_bf16(p, "experts' rows");
  TORCH_CHECK(p.dim() == 3 && p.size(0) == rows && p.size(1) >= 1 &&
              p.size(2) == cols, "experts' rows must be [rows, n, cols]");
  return {p.data_ptr(), 1, (int)p.size(1)};
}

void fused_add_rms_norm(at::Tensor x, at::Tensor residual, at::Tensor weight,
                        double eps, c10::optional<at::Tensor> parts) {
  check_bf16(x, "x"); check_bf16(residual, "residual"); check_bf16(weight, "weight");
  const int H = x.size(-1);
  const long T = x.numel() / H;
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  TORCH_CHECK(!parts.has_value() || (residual.numel() == x.numel() &&
                                     weight.numel() == H),
              "fused_add_rms_norm shapes");
  Addend from{nullptr, 0, 0};
  if (parts.has_value()) from = norm_addend(*parts, T, H);
  fused_add_rms_norm_launch(x.data_ptr(), x.data_ptr(), residual.data_ptr(),
                            weight.data_ptr(), from.data, from.chosen, nullptr,
                            from.n, (float)eps, (int)T, (int)T, H,
                            cur_stream(x));
  HIP_CHECK_LAST();
}

// out = the norm of the rows `pick` of residual + a, a being rows or what
// norm_addend takes
void add_rms_norm_rows(at::Tensor out, at::Tensor a, at::Tensor residual,
                       at::Tensor weight, double eps, at::Tensor pick) {
  check_bf16(out, "out"); check_bf16(residual, "residual");
  check_bf16(weight, "weight");
  const int H = residual.size(-1);
  const long N = residual.numel() / H, T = pick.numel();
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  TORCH_CHECK(pick.is_cuda() && pick.scalar_type() == at::kLong &&
              pick.is_contiguous(), "pick must be int64 on GPU");
  TORCH_CHECK(out.numel() == T * H && weight.numel() == H && N > 0,
              "add_rms_norm_rows shapes");
  Addend from{nullptr, 0, 0};
  if (a.dim() == 3) {
    from = norm_addend(a, N, H);
  } else {
    check_bf16(a, "a");
    TORCH_CHECK(a.numel() == residual.numel(), "add_rms_norm_rows shapes");
  }
  if (T == 0) return;
  fused_add_rms_norm_launch(out.data_ptr(), a.data_ptr(), residual.data_ptr(),
                            weight.data_ptr(), from.data, from.chosen,
                            pick.data_ptr<long>(), from.n, (float)eps, (int)T,
                            (int)N, H, cur_stream(residual));
  HIP_CHECK_LAST();
}

void rotary_embedding(at::Tensor positions, at::Tensor q, at::Tensor k,
                      at::Tensor cos_sin, long head_dim, long rot_dim) {
  const long qs = row_stride_3d(q, "q");
  const long ks = row_stride_3d(k, "k");
  TORCH_CHECK(positions.scalar_type() == at::kLong && positions.is_contiguous());
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous());
  const int T = positions.size(0);
  const int D = (int)head_dim, R = (int)rot_dim;
  const int Hq = q.size(1);
  const int Hk = k.size(1);
  TORCH_CHECK((R / 2) % 8 == 0, "rot_dim/2 must be a multiple of 8");
  rope_neox_launch(positions.data_ptr<long>(), q.data_ptr(), k.data_ptr(),
                   cos_sin.data_ptr<float>(), T, Hq, Hk, D, R, qs, ks,
                   cur_stream(q));
  HIP_CHECK_LAST();
}

void silu_and_mul(at::Tensor out, at::Tensor x) {
  check_bf16(out, "out"); check_bf16(x, "x");
  const int I = out.size(-1);
  const long T = out.numel() / I;
  TORCH_CHECK(x.size(-1) == 2 * I && I % 8 == 0);
  silu_and_mul_launch(out.data_ptr(), x.data_ptr(), T, I, cur_stream(x));
  HIP_CHECK_LAST();
}

void reshape_and_cache(at::Tensor k, at::Tensor v, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor slots) {
  const long ks = row_stride_3d(k, "k");
  const long vs = row_stride_3d(v, "v");
  check_cache(k_cache, "k_cache"); check_cache(v_cache, "v_cache");
  TORCH_CHECK(slots.scalar_type() == at::kLong && slots.is_contiguous());
  const int T = k.size(0), Hkv = k.size(1), D = k.size(2);
  const int BS = k_cache.size(2);
  TORCH_CHECK(k_cache.size(1) == Hkv && k_cache.size(3) == D && D % 8 == 0);
  reshape_and_cache_launch(k.data_ptr(), v.data_ptr(), k_cache.data_ptr(),
                           v_cache.data_ptr(), slots.data_ptr<long>(), T, Hkv,
                           D, BS, ks, vs, is_fp8_cache(k_cache) ? 1 : 0,
                           cur_stream(k));
  HIP_CHECK_LAST();
}

void qkv_store(at::Tensor qkv, long Hq, long Hk,
               c10::optional<at::Tensor> q_norm,
               c10::optional<at::Tensor> k_norm, at::Tensor cos_sin,
               at::Tensor positions, at::Tensor slots, at::Tensor k_cache,
               at::Tensor v_cache, double eps,
               c10::optional<at::Tensor> parts) {
  check_bf16(qkv, "qkv");
  check_cache(k_cache, "k_cache"); check_cache(v_cache, "v_cache");
  const long T = qkv.size(0);
  const int D = k_cache.size(3), BS = k_cache.size(2);
  TORCH_CHECK(qkv.dim() == 2 && qkv.size(1) == (Hq + 2 * Hk) * D
              && k_cache.size(1) == Hk && k_cache.sizes() == v_cache.sizes()
              && k_cache.scalar_type() == v_cache.scalar_type(),
              "qkv_store shapes");
  TORCH_CHECK(positions.is_cuda() && positions.scalar_type() == at::kLong
              && positions.is_contiguous() && positions.numel() == T);
  TORCH_CHECK(slots.is_cuda() && slots.scalar_type() == at::kLong
              && slots.is_contiguous() && slots.numel() == T);
  TORCH_CHECK(cos_sin.is_cuda() && cos_sin.scalar_type() == at::kFloat
              && cos_sin.is_contiguous() && cos_sin.size(1) == D);
  const void* nw[2] = {nullptr, nullptr};
  const c10::optional<at::Tensor>* given[2] = {&q_norm, &k_norm};
  for (int i = 0; i < 2; ++i)
    if (given[i]->has_value()) {
      check_bf16(**given[i], "head norm");
      TORCH_CHECK((*given[i])->numel() == D, "head norm [D]");
      nw[i] = (*given[i])->data_ptr();
    }
  int err = 0;
  qkv_store_launch(qkv.data_ptr(),
                   parts.has_value() ? check_parts(*parts, T, qkv.size(1))
                                     : nullptr,
                   parts.has_value() ? (int)parts->size(0) : 0, nw[0], nw[1], cos_sin.data_ptr<float>(),
                   positions.data_ptr<long>(), slots.data_ptr<long>(),
                   k_cache.data_ptr(), v_cache.data_ptr(), T, (int)Hq,
                   (int)Hk, D, BS, (float)eps, is_fp8_cache(k_cache) ? 1 : 0,
                   &err, cur_stream(qkv));
  TORCH_CHECK(!err, "qkv_store: unsupported head_dim ", D);
  HIP_CHECK_LAST();
}

// host: the words once more, in pinned memory
void greedy_sample(at::Tensor out, at::Tensor logits,
                   c10::optional<at::Tensor> host) {
  check_bf16(logits, "logits");
  TORCH_CHECK(out.scalar_type() == at::kLong && out.is_contiguous());
  const int N = logits.size(0), V = logits.size(1);
  greedy_sample_launch(out.data_ptr<long>(),
                       pinned_words(host, N),
                       logits.data_ptr(), N, V,
                       cur_stream(logits));
  HIP_CHECK_LAST();
}

void mla_decode(at::Tensor ctx_out, at::Tensor q, at::Tensor lat,
                at::Tensor block_tables, at::Tensor seq_lens, double scale) {
  TORCH_CHECK(ctx_out.scalar_type() == at::kFloat && ctx_out.is_contiguous(),
              "ctx_out must be f32 contiguous");
  check_bf16(q, "q"); check_bf16(lat, "lat");
  TORCH_CHECK(q.is_contiguous() && lat.is_contiguous());
  TORCH_CHECK(block_tables.scalar_type() == at::kInt && block_tables.is_contiguous());
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt && seq_lens.is_contiguous());
  const int N = q.size(0), H = q.size(1), LD = q.size(2);
  const int BS = lat.size(2);
  const int R = ctx_out.size(2);
  TORCH_CHECK(lat.size(3) == LD && ctx_out.size(1) == H);
  const int max_blocks = block_tables.size(1);
  int err = 0;
  mla_decode_launch(ctx_out.data_ptr<float>(), q.data_ptr(), lat.data_ptr(),
                    block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(),
                    N, H, R, LD - R, BS, max_blocks, (float)scale, &err,
                    cur_stream(q));
  TORCH_CHECK(!err, "mla_decode: unsupported config R=", R, " LD=", LD,
              " BS=", BS, " H=", H);
  HIP_CHECK_LAST();
}

static const float* sink_ptr_checked(const c10::optional<at::Tensor>& sinks,
                                     int Hq) {
  if (!sinks.has_value()) return nullptr;
  TORCH_CHECK(sinks->scalar_type() == at::kFloat && sinks->is_contiguous()
                  && sinks->numel() == Hq,
              "sinks must be float32 [Hq]");
  return sinks->data_ptr<float>();
}

void paged_attn_decode(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                       at::Tensor v_cache, at::Tensor block_tables,
                       at::Tensor seq_lens, double scale,
                       c10::optional<at::Tensor> sinks, long window,
                       double softcap) {
  check_bf16(out, "out");
  const long qstride = row_stride_3d(q, "q");
  check_cache(k_cache, "k_cache"); check_cache(v_cache, "v_cache");
  TORCH_CHECK(block_tables.scalar_type() == at::kInt && block_tables.is_contiguous());
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt && seq_lens.is_contiguous());
  const int N = q.size(0), Hq = q.size(1), D = q.size(2);
  const int Hkv = k_cache.size(1);
  const int BS = k_cache.size(2);
  TORCH_CHECK(BS == 16, "decode kernel assumes block_size 16");
  const int max_blocks = block_tables.size(1);
  const float* sink_ptr = sink_ptr_checked(sinks, Hq);
  int err = 0;
  const int aligned = ((reinterpret_cast<uintptr_t>(k_cache.data_ptr()) |
                        reinterpret_cast<uintptr_t>(v_cache.data_ptr())) & 15) == 0;
  const DecodeParts parts = decode_parts(N, Hq, Hkv, max_blocks, D,
                                         is_fp8_cache(k_cache) ? 1 : 0,
                                         (int)window, aligned);
  const int nsplit = parts.n;
  // this call's own workspace, from the stream's allocator
  at::Tensor part;
  if (nsplit > 1)
    part = at::empty({(long)N * Hq * nsplit * (D + 2)},
                     out.options().dtype(at::kFloat));
  paged_attn_decode_launch(out.data_ptr(), q.data_ptr(), k_cache.data_ptr(),
                           v_cache.data_ptr(), block_tables.data_ptr<int>(),
                           seq_lens.data_ptr<int>(),
                           nsplit > 1 ? part.data_ptr<float>() : nullptr,
                           parts, N, Hq, Hkv, D, max_blocks,
                           (float)scale, qstride,
                           is_fp8_cache(k_cache) ? 1 : 0, sink_ptr,
                           (int)window, (float)softcap, nullptr, &err, cur_stream(q));
  TORCH_CHECK(!err, "paged_attn_decode: unsupported head_dim/GQ combination: D=",
              D, " Hq=", Hq, " Hkv=", Hkv);
  HIP_CHECK_LAST();
}

// The step's rows from the projection to attention in one launch: qkv_store and
// paged_attn_decode of one row a sequence. rows [N, (Hq + 2 Hkv) D] in bf16, or its fp32
// parts [n, N, ..].
void paged_attn_decode_rows(at::Tensor out, at::Tensor rows, long Hq, long Hkv,
                            c10::optional<at::Tensor> q_norm,
                            c10::optional<at::Tensor> k_norm, at::Tensor cos_sin,
                            at::Tensor positions, at::Tensor slots,
                            at::Tensor k_cache, at::Tensor v_cache,
                            at::Tensor block_tables, at::Tensor seq_lens,
                            double eps, double scale) {
  check_bf16(out, "out");
  check_cache(k_cache, "k_cache"); check_cache(v_cache, "v_cache");
  TORCH_CHECK(out.dim() == 3 && out.size(1) == Hq && Hkv > 0 && Hq % Hkv == 0,
              "out [N, Hq, D]");
  const long N = out.size(0);
  const int D = out.size(2);
  TORCH_CHECK(k_cache.dim() == 4 && k_cache.size(1) == Hkv && k_cache.size(2) == 16 &&
                  k_cache.size(3) == D && k_cache.sizes() == v_cache.sizes() &&
                  k_cache.scalar_type() == v_cache.scalar_type(),
              "pools [blocks, Hkv, 16, D]");
  for (const at::Tensor* t : {&block_tables, &seq_lens})
    TORCH_CHECK(t->is_cuda() && t->scalar_type() == at::kInt && t->is_contiguous(),
                "block_tables and seq_lens are int32");
  for (const at::Tensor* t : {&positions, &slots})
    TORCH_CHECK(t->is_cuda() && t->scalar_type() == at::kLong && t->is_contiguous() &&
                    t->numel() == N, "positions and slots [N]");
  TORCH_CHECK(block_tables.dim() == 2 && block_tables.size(0) == N &&
              block_tables.size(1) > 0 && seq_lens.numel() == N);
  TORCH_CHECK(cos_sin.is_cuda() && cos_sin.scalar_type() == at::kFloat
              && cos_sin.is_contiguous() && cos_sin.size(1) == D);
  const long W = (Hq + 2 * Hkv) * D;
  NewRows nr{};
  if (rows.dim() == 3) {
    nr.parts = check_parts(rows, N, W);
    nr.nparts = (int)rows.size(0);
  } else {
    check_bf16(rows, "rows");
    TORCH_CHECK(rows.dim() == 2 && rows.size(0) == N && rows.size(1) == W &&
                    at_16(rows), "rows [N, (Hq + 2 Hkv) D]");
    nr.rows = (const unsigned short*)rows.data_ptr();
  }
  const c10::optional<at::Tensor>* given[2] = {&q_norm, &k_norm};
  const unsigned short** norms[2] = {&nr.q_norm, &nr.k_norm};
  for (int i = 0; i < 2; ++i)
    if (given[i]->has_value()) {
      check_bf16(**given[i], "head norm");
      TORCH_CHECK((*given[i])->numel() == D && at_16(**given[i]), "head norm [D]");
      *norms[i] = (const unsigned short*)(*given[i])->data_ptr();
    }
  nr.cos_sin = cos_sin.data_ptr<float>();
  nr.positions = positions.data_ptr<long>();
  nr.slots = slots.data_ptr<long>();
  nr.eps = (float)eps;
  const int fp8 = is_fp8_cache(k_cache) ? 1 : 0;
  const int max_blocks = block_tables.size(1);
  const DecodeParts parts = decode_parts(N, Hq, Hkv, max_blocks, D, fp8, 0,
                                         at_16(k_cache) && at_16(v_cache));
  at::Tensor part;
  if (parts.n > 1)
    part = at::empty({N * Hq * parts.n * (D + 2)}, out.options().dtype(at::kFloat));
  int err = 0;
  paged_attn_decode_launch(out.data_ptr(), nullptr, k_cache.data_ptr(),
                           v_cache.data_ptr(), block_tables.data_ptr<int>(),
                           seq_lens.data_ptr<int>(),
                           parts.n > 1 ? part.data_ptr<float>() : nullptr, parts, N,
                           Hq, Hkv, D, max_blocks, (float)scale, 0, fp8, nullptr, 0,
                           0.f, &nr, &err, cur_stream(out));
  TORCH_CHECK(!err, "paged_attn_decode_rows: D=", D, " Hq=", Hq, " Hkv=", Hkv);
  HIP_CHECK_LAST();
}

void flash_prefill(at::Tensor out, at::Tensor q, at::Tensor k, at::Tensor v,
                   at::Tensor tile_start, at::Tensor tile_q0,
                   at::Tensor tile_len, double scale,
                   c10::optional<at::Tensor> sinks, long window,
                   double softcap) {
  check_bf16(out, "out");
  const long qs = row_stride_3d(q, "q");
  const long ks = row_stride_3d(k, "k");
  const long vs = row_stride_3d(v, "v");
  TORCH_CHECK(tile_start.scalar_type() == at::kInt && tile_start.is_contiguous());
  const int ntiles = tile_start.size(0);
  const int Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
  const int DV = out.size(2);  // value dim (== D except MLA 192/128)
  TORCH_CHECK(v.size(2) == DV, "v/out value dims must match");
  int err = 0;
  flash_prefill_launch(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                       tile_start.data_ptr<int>(), tile_q0.data_ptr<int>(),
                       tile_len.data_ptr<int>(), ntiles, Hq, Hkv, D, DV,
                       (float)scale, qs, ks, vs, sink_ptr_checked(sinks, Hq),
                       (int)window, (float)softcap, &err, cur_stream(q));
  TORCH_CHECK(!err, "flash_prefill: unsupported config D=", D, " DV=", DV);
  HIP_CHECK_LAST();
}

void flash_prefill_paged(at::Tensor out, at::Tensor q, at::Tensor k_cache,
                         at::Tensor v_cache, at::Tensor block_tables,
                         at::Tensor tile_qstart, at::Tensor tile_q0,
                         at::Tensor tile_hist, at::Tensor tile_new,
                         at::Tensor tile_seq, double scale,
                         c10::optional<at::Tensor> sinks, long window,
                         double softcap) {
  check_bf16(out, "out");
  const long qs = row_stride_3d(q, "q");
  check_bf16(k_cache, "k_cache"); check_bf16(v_cache, "v_cache");
  for (auto* t : {&block_tables, &tile_qstart, &tile_q0, &tile_hist,
                  &tile_new, &tile_seq}) {
    TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous());
  }
  const int ntiles = tile_qstart.size(0);
  const int Hq = q.size(1), D = q.size(2);
  const int Hkv = k_cache.size(1);
  TORCH_CHECK(k_cache.size(2) == 16, "paged prefill assumes block_size 16");
  const int maxb = block_tables.size(1);
  int err = 0;
  flash_prefill_paged_launch(
      out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
      block_tables.data_ptr<int>(), tile_qstart.data_ptr<int>(),
      tile_q0.data_ptr<int>(), tile_hist.data_ptr<int>(),
      tile_new.data_ptr<int>(), tile_seq.data_ptr<int>(), ntiles, Hq, Hkv, D,
      maxb, (float)scale, qs, sink_ptr_checked(sinks, Hq), (int)window,
      (float)softcap, &err, cur_stream(q));
  TORCH_CHECK(!err, "flash_prefill_paged: unsupported config D=", D);
  HIP_CHECK_LAST();
}

void gemm8(at::Tensor out, at::Tensor x, at::Tensor w, long safe) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(w, "w");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  int err = 0;
  gemm8_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K,
               (int)safe, &err, cur_stream(x));
  TORCH_CHECK(!err, "gemm8: unsupported shape M=", M, " N=", N, " K=", K,
              " (need N%256==0, K%128==0)");
  HIP_CHECK_LAST();
}

void skinny_gemm(at::Tensor out, at::Tensor x, at::Tensor w,
                 c10::optional<at::Tensor> workspace, long splitk,
                 long version) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(w, "w");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(N % 128 == 0, "N must be a multiple of 128");
  TORCH_CHECK(K % (64 * splitk) == 0, "K must be a multiple of 64*splitk");
  void* ws = nullptr;
  if (splitk > 1) {
    TORCH_CHECK(workspace.has_value(), "splitk>1 needs an f32 workspace");
    TORCH_CHECK(workspace->scalar_type() == at::kFloat &&
                workspace->numel() >= (long)splitk * M * N);
    ws = workspace->data_ptr();
  }
  if (version == 2) {
    TORCH_CHECK(N % 256 == 0, "v2 needs N % 256 == 0");
    skinny_gemm_v2_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), ws, M,
                          N, K, (int)splitk, cur_stream(x));
  } else {
    skinny_gemm_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), ws, M, N,
                       K, (int)splitk, cur_stream(x));
  }
  HIP_CHECK_LAST();
}

void moe_down_scale(at::Tensor contrib, at::Tensor act, at::Tensor w,
                    at::Tensor offs, at::Tensor counts, at::Tensor order,
                    at::Tensor flat_w, c10::optional<at::Tensor> bias,
                    c10::optional<at::Tensor> tiles,
                    c10::optional<at::Tensor> ntiles) {
  check_bf16(contrib, "contrib"); check_bf16(act, "act"); check_bf16(w, "w");
  for (auto* t : {&offs, &counts, &order}) {
    TORCH_CHECK(t->scalar_type() == at::kInt && t->is_contiguous());
  }
  TORCH_CHECK(flat_w.scalar_type() == at::kFloat && flat_w.is_contiguous());
  const int E = w.size(0), H = w.size(1), I = w.size(2);
  TORCH_CHECK(act.size(1) == I && contrib.size(1) == H);
  TORCH_CHECK(contrib.size(0) == order.size(0));
  const void* bias_ptr = nullptr;
  if (bias.has_value()) {
    check_bf16(*bias, "bias");
    TORCH_CHECK(bias->numel() == (long)E * H, "down bias must be [E, H]");
    bias_ptr = bias->data_ptr();
  }
  const int *list = nullptr, *n = nullptr;
  if (tiles.has_value() && ntiles.has_value()) {
    check_i32(*tiles, 2 * (contrib.size(0) / 128 + E), "tiles");
    check_i32(*ntiles, 1, "ntiles");
    list = tiles->data_ptr<int>();
    n = ntiles->data_ptr<int>();
  }
  int err = 0;
  moe_down_scale_launch(contrib.data_ptr(), act.data_ptr(), w.data_ptr(),
                        offs.data_ptr<int>(), counts.data_ptr<int>(),
                        order.data_ptr<int>(), flat_w.data_ptr<float>(),
                        bias_ptr, list, n, contrib.size(0), E, H, I, &err, cur_stream(act));
  TORCH_CHECK(!err, "moe_down_scale: unsupported dims H=", H, " I=", I);
  HIP_CHECK_LAST();
}

void moe_topk(at::Tensor experts, at::Tensor weights, at::Tensor logits,
              bool renorm) {
  const int parts = logits.dim() == 3 ? logits.size(0) : 1;
  const int T = logits.size(-2), E = logits.size(-1), k = experts.size(1);
  check_i32(experts, (long)T * k, "experts");
  TORCH_CHECK(logits.is_cuda() && logits.scalar_type() == at::kFloat
              && logits.is_contiguous(), "logits must be fp32");
  TORCH_CHECK(weights.is_cuda() && weights.scalar_type() == at::kFloat
              && weights.is_contiguous()
              && weights.numel() == (long)T * k
              && experts.numel() == (long)T * k, "experts / weights [T, k]");
  int err = 0;
  moe_topk_launch(experts.data_ptr<int>(), weights.data_ptr<float>(),
                  logits.data_ptr<float>(), T, E, k, renorm ? 1 : 0, parts,
                  &err, cur_stream(logits));
  TORCH_CHECK(!err, "moe_topk: unsupported E=", E, " k=", k);
  HIP_CHECK_LAST();
}

void moe_route(at::Tensor experts, at::Tensor weights, at::Tensor x,
               at::Tensor w, bool renorm) {
  check_bf16(x, "x"); check_bf16(w, "w");
  const int T = x.size(0), H = x.size(1), E = w.size(0), k = experts.size(1);
  check_i32(experts, (long)T * k, "experts");
  TORCH_CHECK(w.size(1) == H && (uintptr_t)x.data_ptr() % 16 == 0
              && (uintptr_t)w.data_ptr() % 16 == 0, "moe_route operands");
  TORCH_CHECK(weights.is_cuda() && weights.scalar_type() == at::kFloat
              && weights.is_contiguous()
              && weights.numel() == (long)T * k
              && experts.numel() == (long)T * k, "experts / weights [T, k]");
  int err = 0;
  moe_route_launch(experts.data_ptr<int>(), weights.data_ptr<float>(),
                   x.data_ptr(), w.data_ptr(), T, E, H, k, renorm ? 1 : 0,
                   &err, cur_stream(x));
  TORCH_CHECK(!err, "moe_route: unsupported E=", E, " H=", H, " k=", k);
  HIP_CHECK_LAST();
}

// -> (order, s_tok, counts, offs, tiles, ntiles), and the weights in the order of the
// sorted rows where they are given
std::vector<at::Tensor> moe_sort(at::Tensor experts, long E, long k,
                                 c10::optional<at::Tensor> weights) {
  const long TK = experts.numel();
  check_i32(experts, TK, "experts");
  at::Tensor s_w;
  if (weights.has_value()) {
    TORCH_CHECK(weights->is_cuda() && weights->scalar_type() == at::kFloat &&
                weights->is_contiguous() && weights->numel() == TK,
                "weights [TK] fp32");
    s_w = at::empty({TK}, weights->options());
  }
  TORCH_CHECK(TK < (1L << 30) && k >= 1 && E >= 1, "moe_sort sizes");
  auto o = experts.options();
  at::Tensor order = at::empty({TK}, o), s_tok = at::empty({TK}, o);
  at::Tensor counts = at::empty({E}, o), offs = at::empty({E}, o);
  at::Tensor tiles = at::empty({TK / 128 + E, 2}, o), n = at::empty({1}, o);
  const long slices = moe_sort_slices((int)TK);
  at::Tensor hist = at::empty({slices * E}, o);
  int err = 0;
  moe_sort_launch(order.data_ptr<int>(), s_tok.data_ptr<int>(),
                  s_w.defined() ? s_w.data_ptr<float>() : nullptr,
                  s_w.defined() ? weights->data_ptr<float>() : nullptr,
                  counts.data_ptr<int>(), offs.data_ptr<int>(),
                  tiles.data_ptr<int>(), n.data_ptr<int>(),
                  hist.data_ptr<int>(), experts.data_ptr<int>(), (int)TK, (int)E, (int)k, &err,
                  cur_stream(experts));
  TORCH_CHECK(!err, "moe_sort: unsupported E=", E);
  HIP_CHECK_LAST();
  if (s_w.defined()) return {order, s_tok, counts, offs, tiles, n, s_w};
  return {order, s_tok, counts, offs, tiles, n};
}

// moe_topk and moe_sort (without weights) in one launch: what moe_sort returns
std::vector<at::Tensor> moe_choose(at::Tensor experts, at::Tensor weights,
                                   at::Tensor logits, bool renorm) {
  const int parts = logits.dim() == 3 ? logits.size(0) : 1;
  const int T = logits.size(-2), E = logits.size(-1), k = experts.size(1);
  check_i32(experts, (long)T * k, "experts");
  TORCH_CHECK(logits.is_cuda() && logits.scalar_type() == at::kFloat
              && logits.is_contiguous(), "logits must be fp32");
  TORCH_CHECK(weights.is_cuda() && weights.scalar_type() == at::kFloat
              && weights.is_contiguous()
              && weights.numel() == (long)T * k
              && experts.numel() == (long)T * k, "experts / weights [T, k]");
  const long TK = (long)T * k;
  auto o = experts.options();
  at::Tensor order = at::empty({TK}, o), s_tok = at::empty({TK}, o);
  at::Tensor counts = at::empty({E}, o), offs = at::empty({E}, o);
  at::Tensor tiles = at::empty({TK / 128 + E, 2}, o), n = at::empty({1}, o);
  int err = 0;
  moe_choose_launch(experts.data_ptr<int>(), weights.data_ptr<float>(),
                    order.data_ptr<int>(), s_tok.data_ptr<int>(),
                    counts.data_ptr<int>(), offs.data_ptr<int>(),
                    tiles.data_ptr<int>(), n.data_ptr<int>(),
                    logits.data_ptr<float>(), T, E, k, renorm ? 1 : 0, parts, &err,
                    cur_stream(logits));
  TORCH_CHECK(!err, "moe_choose: unsupported T=", T, " E=", E, " k=", k);
  HIP_CHECK_LAST();
  return {order, s_tok, counts, offs, tiles, n};
}

// moe_tile without bias or another activation, in tiles of up to 320 rows; s_w: the
// weights that moe_sort sorted
void moe_wide(bool down, at::Tensor out, at::Tensor src, at::Tensor w,
              at::Tensor rows, at::Tensor offs, at::Tensor counts,
              c10::optional<at::Tensor> s_w) {
  check_bf16(out, "out"); check_bf16(src, "src"); check_bf16(w, "w");
  TORCH_CHECK(w.dim() == 3 && src.dim() == 2 && out.dim() == 2, "moe_wide shapes");
  const long E = w.size(0), K = w.size(2), TK = out.size(0);
  const long N = down ? w.size(1) : w.size(1) / 2;
  check_i32(rows, TK, "rows");
  check_i32(offs, E, "offs");
  check_i32(counts, E, "counts");
  TORCH_CHECK(src.size(1) == K && out.size(1) == N &&
              w.size(1) == (down ? N : 2 * N) && (!down || src.size(0) == TK),
              "moe_wide shapes");
  TORCH_CHECK((uintptr_t)src.data_ptr() % 16 == 0 &&
              (uintptr_t)w.data_ptr() % 16 == 0 &&
              (uintptr_t)out.data_ptr() % 16 == 0, "moe_wide addresses");
  const float* sw = nullptr;
  if (down) {
    TORCH_CHECK(s_w.has_value() && s_w->is_cuda() &&
                s_w->scalar_type() == at::kFloat && s_w->is_contiguous() &&
                s_w->numel() == TK, "s_w [TK] fp32");
    sw = s_w->data_ptr<float>();
  }
  TORCH_CHECK(N < (1l << 30) && K < (1l << 30) &&
              moe_wide_takes(down ? 1 : 0, src.size(0), TK, (int)E, (int)N, (int)K),
              "moe_wide: unsupported E=", E, " N=", N, " K=", K);
  moe_wide_launch(down ? 1 : 0, out.data_ptr(), src.data_ptr(), w.data_ptr(),
                  rows.data_ptr<int>(), sw, offs.data_ptr<int>(),
                  counts.data_ptr<int>(), src.size(0), TK, (int)E, (int)N, (int)K,
                  cur_stream(src));
  HIP_CHECK_LAST();
}

void moe_sum(at::Tensor out, at::Tensor contrib, long k) {
  check_bf16(out, "out"); check_bf16(contrib, "contrib");
  const long T = out.size(0);
  const int H = out.size(1);
  TORCH_CHECK(H % 8 == 0 && contrib.numel() == T * k * H, "moe_sum shapes");
  moe_sum_launch(out.data_ptr(), contrib.data_ptr(), T, (int)k, H,
                 cur_stream(out));
  HIP_CHECK_LAST();
}

// down: contrib[rows[j]] = (src[j] @ w[e]^T + bias) * flat_w[rows[j]];
// else act[j] = act(src[rows[j]] @ gate^T, ... @ up^T), over the tile list
void moe_tile(bool down, at::Tensor out, at::Tensor src, at::Tensor w,
              at::Tensor rows, at::Tensor tiles, at::Tensor ntiles,
              at::Tensor offs, at::Tensor counts,
              c10::optional<at::Tensor> flat_w,
              c10::optional<at::Tensor> bias, long act_mode) {
  check_bf16(out, "out"); check_bf16(src, "src"); check_bf16(w, "w");
  const int E = w.size(0), K = w.size(2);
  const long N = down ? w.size(1) : w.size(1) / 2;
  check_i32(rows, out.size(0), "rows");
  check_i32(ntiles, 1, "ntiles");
  check_i32(offs, E, "offs");
  check_i32(counts, E, "counts");
  check_i32(tiles, 2 * (out.size(0) / 128 + E), "tiles");
  TORCH_CHECK(src.size(1) == K && out.size(1) == N, "moe_tile shapes");
  TORCH_CHECK(!down || src.size(0) == out.size(0), "moe_tile rows");
  const float* fw = nullptr;
  if (down) {
    TORCH_CHECK(flat_w.has_value() && flat_w->is_cuda()
                && flat_w->scalar_type() == at::kFloat
                && flat_w->is_contiguous()
                && flat_w->numel() == out.size(0), "flat_w [TK] fp32");
    fw = flat_w->data_ptr<float>();
  }
  const void* bias_ptr = nullptr;
  if (bias.has_value()) {
    check_bf16(*bias, "bias");
    TORCH_CHECK(bias->numel() == (long)E * w.size(1), "bias shape");
    bias_ptr = bias->data_ptr();
  }
  int err = 0;
  moe_tile_launch(down ? 1 : 0, out.data_ptr(), src.data_ptr(), w.data_ptr(),
                  rows.data_ptr<int>(), tiles.data_ptr<int>(),
                  ntiles.data_ptr<int>(), offs.data_ptr<int>(),
                  counts.data_ptr<int>(), fw, bias_ptr, (int)act_mode, src.size(0),
                  (int)(out.size(0) / 128 + E), (int)N, K, &err,
                  cur_stream(src));
  TORCH_CHECK(!err, "moe_tile: unsupported dims N=", N, " K=", K);
  HIP_CHECK_LAST();
}

// moe_tile without bias or another activation, for few rows an expert
void moe_few(bool down, at::Tensor out, at::Tensor src, at::Tensor w,
             at::Tensor rows, at::Tensor tiles, at::Tensor ntiles,
             at::Tensor offs, at::Tensor counts,
             c10::optional<at::Tensor> flat_w) {
  check_bf16(out, "out"); check_bf16(src, "src"); check_bf16(w, "w");
  TORCH_CHECK(w.dim() == 3 && src.dim() == 2 && out.dim() == 2, "moe_few shapes");
  const long E = w.size(0), K = w.size(2), TK = out.size(0);
  const long N = down ? w.size(1) : w.size(1) / 2;
  check_i32(rows, TK, "rows");
  check_i32(ntiles, 1, "ntiles");
  check_i32(offs, E, "offs");
  check_i32(counts, E, "counts");
  check_i32(tiles, 2 * (TK / 128 + E), "tiles");
  TORCH_CHECK(src.size(1) == K && out.size(1) == N &&
              w.size(1) == (down ? N : 2 * N) && (!down || src.size(0) == TK),
              "moe_few shapes");
  TORCH_CHECK((uintptr_t)src.data_ptr() % 16 == 0 &&
              (uintptr_t)w.data_ptr() % 16 == 0, "moe_few addresses");
  const float* fw = nullptr;
  if (down) {
    TORCH_CHECK(flat_w.has_value() && flat_w->is_cuda() &&
                flat_w->scalar_type() == at::kFloat && flat_w->is_contiguous() &&
                flat_w->numel() == TK, "flat_w [TK] fp32");
    fw = flat_w->data_ptr<float>();
  }
  int err = 0;
  moe_few_launch(down ? 1 : 0, out.data_ptr(), src.data_ptr(), w.data_ptr(),
                 rows.data_ptr<int>(), tiles.data_ptr<int>(),
                 ntiles.data_ptr<int>(), offs.data_ptr<int>(),
                 counts.data_ptr<int>(), fw, src.size(0), TK, (int)E, (int)N,
                 (int)K, &err, cur_stream(src));
  TORCH_CHECK(!err, "moe_few: unsupported dims N=", N, " K=", K);
  HIP_CHECK_LAST();
}

// fp32 parts [splits, M, N] of the product, not added up
at::Tensor rows_tile_parts(at::Tensor x, at::Tensor w, long cols, long splits) {
  check_bf16(w, "w");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() == 2
              && x.stride(1) == 1 && x.stride(0) % 8 == 0, "x rows of bf16");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && (uintptr_t)x.data_ptr() % 16 == 0 &&
              (uintptr_t)w.data_ptr() % 16 == 0, "rows_tile_parts shapes");
  at::Tensor parts = at::empty({splits, M, N}, x.options().dtype(at::kFloat));
  int err = 0;
  rows_tile_launch(nullptr, parts.data_ptr(), x.data_ptr(), w.data_ptr(), M, N,
                   K, x.stride(0), (int)cols, (int)splits, 0, &err,
                   cur_stream(x));
  TORCH_CHECK(!err, "rows_tile_parts: unsupported M=", M, " N=", N, " K=", K);
  HIP_CHECK_LAST();
  return parts;
}

// silu: w holds the gate's rows and behind them the up product's, out is
// silu(gate) * up
void rows_tile(at::Tensor out, at::Tensor x, at::Tensor w, long cols,
               long splits, bool silu) {
  check_bf16(out, "out"); check_bf16(w, "w");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() == 2
              && x.stride(1) == 1 && x.stride(0) % 8 == 0
              && (uintptr_t)x.data_ptr() % 16 == 0, "x rows of bf16");
  const int M = x.size(0), K = x.size(1), N = out.size(1);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M &&
              w.size(0) == (silu ? 2l * N : N) &&
              (uintptr_t)w.data_ptr() % 16 == 0, "rows_tile shapes");
  at::Tensor parts;
  if (splits > 1)
    parts = at::empty({splits, M, N}, out.options().dtype(at::kFloat));
  int err = 0;
  rows_tile_launch(out.data_ptr(), splits > 1 ? parts.data_ptr() : nullptr,
                   x.data_ptr(), w.data_ptr(), M, N, K, x.stride(0),
                   (int)cols, (int)splits, silu ? 1 : 0, &err, cur_stream(x));
  TORCH_CHECK(!err, "rows_tile: unsupported M=", M, " N=", N, " K=", K);
  HIP_CHECK_LAST();
}

void rows_gemm(at::Tensor out, at::Tensor x, at::Tensor w) {
  check_bf16(out, "out"); check_bf16(w, "w");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() == 2
              && x.stride(1) == 1 && x.stride(0) % 8 == 0
              && (uintptr_t)x.data_ptr() % 16 == 0, "x rows of bf16");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N,
              "rows_gemm shapes");
  int err = 0;
  rows_gemm_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K,
                   x.stride(0), &err, cur_stream(x));
  TORCH_CHECK(!err, "rows_gemm: unsupported M=", M, " K=", K);
  HIP_CHECK_LAST();
}

// operands of a product of many rows -> M, N weight rows, K
void check_wide(const at::Tensor& x, const at::Tensor& w) {
  check_bf16(w, "w");
  TORCH_CHECK(x.is_cuda() && x.scalar_type() == at::kBFloat16 && x.dim() == 2
              && x.stride(1) == 1 && x.stride(0) % 8 == 0
              && (uintptr_t)x.data_ptr() % 16 == 0, "x rows of bf16");
  TORCH_CHECK(w.dim() == 2 && w.size(1) == x.size(1) &&
              (uintptr_t)w.data_ptr() % 16 == 0 && x.size(0) < (1l << 31) &&
              w.size(0) < (1l << 30) && x.size(1) < (1l << 30), "wide shapes");
}

// out = x w^T of many rows in tiles of 32 rf x 32 cf; silu: silu(gate) * up, w holding
// the gate's rows and behind them the up product's
void wide_rows(at::Tensor out, at::Tensor x, at::Tensor w, int64_t rf, int64_t cf,
               bool silu) {
  check_bf16(out, "out");
  check_wide(x, w);
  const long M = x.size(0), N = out.size(1), K = x.size(1);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == M && w.size(0) == (silu ? 2 : 1) * N &&
              (uintptr_t)out.data_ptr() % 16 == 0, "wide_rows shapes");
  TORCH_CHECK(rf >= 0 && rf <= 9 && cf >= 0 && cf <= 9, "wide_rows tiles");
  int err = 0;
  wide_launch(silu ? 0 : 1, out.data_ptr(), x.data_ptr(), w.data_ptr(), (int)M, (int)N,
              (int)K, x.stride(0), 1, (int)rf, (int)cf, &err, cur_stream(x));
  TORCH_CHECK(!err, "wide_rows: unsupported M=", M, " N=", N, " K=", K, " tiles ", rf,
              " x ", cf);
  HIP_CHECK_LAST();
}

// fp32 parts [splits, M, N] of the product, not added up
at::Tensor wide_parts(at::Tensor x, at::Tensor w, int64_t splits, int64_t rf,
                      int64_t cf) {
  check_wide(x, w);
  TORCH_CHECK(rf >= 0 && rf <= 9 && cf >= 0 && cf <= 9, "wide_parts tiles");
  const long M = x.size(0), N = w.size(0), K = x.size(1);
  TORCH_CHECK(splits >= 1 && splits <= K / 128, "wide_parts: parts of K=", K);
  at::Tensor parts = at::empty({splits, M, N}, x.options().dtype(at::kFloat));
  int err = 0;
  wide_launch(2, parts.data_ptr(), x.data_ptr(), w.data_ptr(), (int)M, (int)N, (int)K,
              x.stride(0), (int)splits, (int)rf, (int)cf, &err, cur_stream(x));
  TORCH_CHECK(!err, "wide_parts: unsupported M=", M, " N=", N, " K=", K, " tiles ", rf,
              " x ", cf);
  HIP_CHECK_LAST();
  return parts;
}

// the up product from counts and offsets that the caller sorted by
void moe_gate_up_silu(at::Tensor act, at::Tensor x, at::Tensor w,
                      at::Tensor s_tok, at::Tensor offs, at::Tensor counts,
                      c10::optional<at::Tensor> bias, long act_mode) {
  const int E = w.size(0);
  const long most = act.size(0) / 128 + E;
  check_i32(counts, E, "counts");
  TORCH_CHECK(act.size(0) == s_tok.size(0));
  at::Tensor tiles = at::empty({most, 2}, counts.options());
  at::Tensor n = at::empty({1}, counts.options());
  moe_tiles_launch(tiles.data_ptr<int>(), n.data_ptr<int>(),
                   counts.data_ptr<int>(), E, (int)most, cur_stream(x));
  moe_tile(false, act, x, w, s_tok, tiles, n, offs, counts, c10::nullopt,
           bias, act_mode);
}

// operands of a packed product
void check_w4(const at::Tensor& x, const at::Tensor& qw, const at::Tensor& sc,
              const at::Tensor& zs) {
  check_bf16(x, "x"); check_bf16(sc, "sc"); check_bf16(zs, "zs");
  TORCH_CHECK(qw.scalar_type() == at::kByte && qw.is_contiguous());
  const int K = x.size(1), N = qw.size(0);
  TORCH_CHECK(qw.size(1) == K / 2);
  TORCH_CHECK(sc.size(0) == N && sc.size(1) == K / 128);
}


void w4_gemm(at::Tensor out, at::Tensor x, at::Tensor qw, at::Tensor sc,
             at::Tensor zs) {
  check_bf16(out, "out");
  check_w4(x, qw, sc, zs);
  const int M = x.size(0), K = x.size(1), N = qw.size(0);
  TORCH_CHECK(out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(w4_has(N, K), "w4_gemm: unsupported shape M=", M, " N=", N, " K=",
              K, " (need N%64==0, K%128==0)");
  const hipStream_t s = cur_stream(x);
  // the rows' form takes operands at any address
  if (w4_by_rows(M, N, K) || !at_16(x) || !at_16(qw) || !at_16(out)) {
    w4_rows_launch(out.data_ptr(), x.data_ptr(), qw.data_ptr(), sc.data_ptr(),
                   zs.data_ptr(), M, N, K, s);
  } else if (const int splits = w4_splits(M, N, K); splits > 1) {
    at::Tensor parts = at::empty({splits, M, N}, x.options().dtype(at::kFloat));
    w4_parts_launch(parts.data_ptr<float>(), x.data_ptr(), qw.data_ptr(),
                    sc.data_ptr(), zs.data_ptr(), M, N, K, splits, s);
    rows_join_launch(out.data_ptr(), parts.data_ptr<float>(), (long)M * N, splits,
                     s);
  } else {
    w4_tile_launch(out.data_ptr(), x.data_ptr(), qw.data_ptr(), sc.data_ptr(),
                   zs.data_ptr(), M, N, K, s);
  }
  HIP_CHECK_LAST();
}

// fp32 parts [n, M, N] of the product, not added up, or none where it is not cut
c10::optional<at::Tensor> w4_parts(at::Tensor x, at::Tensor qw, at::Tensor sc,
                                   at::Tensor zs) {
  check_w4(x, qw, sc, zs);
  const int M = x.size(0), K = x.size(1), N = qw.size(0);
  if (!w4_has(N, K) || !w4_cuts(M, N, K) || !at_16(x) || !at_16(qw))
    return c10::nullopt;
  const int splits = w4_splits(M, N, K);
  at::Tensor parts = at::empty({splits, M, N}, x.options().dtype(at::kFloat));
  w4_parts_launch(parts.data_ptr<float>(), x.data_ptr(), qw.data_ptr(),
                  sc.data_ptr(), zs.data_ptr(), M, N, K, splits, cur_stream(x));
  HIP_CHECK_LAST();
  return parts;
}

// silu(gate) * up of the product, qw holding the gate's rows and behind them the
// up product's; none where there is no such form (w4_silu_wins says where it is the
// faster one)
c10::optional<at::Tensor> w4_silu(at::Tensor x, at::Tensor qw, at::Tensor sc,
                                  at::Tensor zs) {
  check_w4(x, qw, sc, zs);
  const int M = x.size(0), K = x.size(1), N = qw.size(0);
  if (!w4_has(N, K) || N % 128 != 0 || !at_16(x) || !at_16(qw))
    return c10::nullopt;
  at::Tensor out = at::empty({M, N / 2}, x.options());
  w4_silu_launch(out.data_ptr(), x.data_ptr(), qw.data_ptr(), sc.data_ptr(),
                 zs.data_ptr(), M, N / 2, K, cur_stream(x));
  HIP_CHECK_LAST();
  return out;
}

void w4_dequant(at::Tensor out, at::Tensor qw, at::Tensor sc, at::Tensor zs) {
  check_bf16(out, "out"); check_bf16(sc, "sc"); check_bf16(zs, "zs");
  TORCH_CHECK(qw.scalar_type() == at::kByte && qw.is_contiguous());
  const long N = qw.size(0);
  const int K = (int)(qw.size(1) * 2);
  TORCH_CHECK(out.size(0) == N && out.size(1) == K);
  int err = 0;
  w4_dequant_launch(out.data_ptr(), qw.data_ptr(), sc.data_ptr(),
                    zs.data_ptr(), N, K, &err, cur_stream(out));
  TORCH_CHECK(!err, "w4_dequant: K must be a multiple of 128");
  HIP_CHECK_LAST();
}

void gemm_lab(at::Tensor out, at::Tensor x, at::Tensor w, long mode) {
  check_bf16(out, "out"); check_bf16(x, "x"); check_bf16(w, "w");
  const int M = x.size(0), K = x.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  int err = 0;
  gemm_lab_launch(out.data_ptr(), x.data_ptr(), w.data_ptr(), M, N, K,
                  (int)mode, &err, cur_stream(x));
  TORCH_CHECK(!err, "gemm_lab: unsupported shape/mode M=", M, " N=", N,
              " K=", K, " mode=", mode);
  HIP_CHECK_LAST();
}

at::Tensor mfma_probe(at::Tensor a, at::Tensor b) {
  check_bf16(a, "a"); check_bf16(b, "b");
  auto d = at::zeros({16, 16}, a.options().dtype(at::kFloat));
  mfma_probe_launch(d.data_ptr<float>(), a.data_ptr(), b.data_ptr(),
                    cur_stream(a));
  HIP_CHECK_LAST();
  return d;
}

}  // namespace

#undef HIP_CHECK_LAST
PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "RMSNorm (bf16)");
  m.def("fused_add_rms_norm", &fused_add_rms_norm,
        "residual+=x (or the sum of parts); x=norm(residual)*w", py::arg("x"),
        py::arg("residual"), py::arg("weight"), py::arg("eps"),
        py::arg("parts") = py::none());
  m.def("embed_rms_norm", &embed_rms_norm, "rows of tokens and their RMS norm");
  m.def("add_rms_norm_rows", &add_rms_norm_rows,
        "RMS norm of picked rows of residual + a");
  m.def("rotary_embedding", &rotary_embedding, "in-place neox RoPE on q,k");
  m.def("silu_and_mul", &silu_and_mul, "silu(x[:d])*x[d:]");
  m.def("reshape_and_cache", &reshape_and_cache, "scatter K/V into paged pool");
  m.def("qkv_store", &qkv_store,
        "head norms, rotation in place and cache write of a q|k|v row",
        py::arg("qkv"), py::arg("q_heads"), py::arg("kv_heads"),
        py::arg("q_norm"), py::arg("k_norm"), py::arg("cos_sin"),
        py::arg("positions"), py::arg("slots"), py::arg("k_cache"),
        py::arg("v_cache"), py::arg("eps"), py::arg("parts") = py::none());
  m.def("greedy_sample", &greedy_sample, "argmax over vocab", py::arg("out"),
        py::arg("logits"), py::arg("host") = py::none());
  m.def("mla_decode", &mla_decode,
        "MLA absorbed decode over the paged latent cache (DeepSeek)");
  m.def("paged_attn_decode_rows", &paged_attn_decode_rows,
        "head norms, rotation, cache write and paged attention of a step's rows");
  m.def("paged_attn_decode", &paged_attn_decode, "paged GQA decode attention",
        py::arg("out"), py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_tables"), py::arg("seq_lens"), py::arg("scale"),
        py::arg("sinks") = py::none(), py::arg("window") = 0,
        py::arg("softcap") = 0.0);
  m.def("flash_prefill", &flash_prefill, "varlen causal MFMA prefill attention",
        py::arg("out"), py::arg("q"), py::arg("k"), py::arg("v"),
        py::arg("tile_start"), py::arg("tile_q0"), py::arg("tile_len"),
        py::arg("scale"), py::arg("sinks") = py::none(),
        py::arg("window") = 0, py::arg("softcap") = 0.0);
  m.def("flash_prefill_paged", &flash_prefill_paged,
        py::arg("out"), py::arg("q"), py::arg("k_cache"), py::arg("v_cache"),
        py::arg("block_tables"), py::arg("tile_qstart"), py::arg("tile_q0"),
        py::arg("tile_hist"), py::arg("tile_new"), py::arg("tile_seq"),
        py::arg("scale"), py::arg("sinks") = py::none(),
        py::arg("window") = 0, py::arg("softcap") = 0.0,
        "MFMA prefill attention with paged-KV history (suffix/chunk rows)");
  m.def("mfma_probe", &mfma_probe, "16x16x32 bf16 MFMA layout probe");
  m.def("skinny_gemm", &skinny_gemm, "split-K skinny GEMM (bf16, f32 accum)");
  m.def("gemm8", &gemm8, "8-phase pipelined 256x256 GEMM (bf16, f32 accum)");
  m.def("gemm_lab", &gemm_lab, "GEMM schedule lab variants (A/B vs hipBLASLt)");
  m.def("rows_tile_parts", &rows_tile_parts,
        "fp32 parts over k of a bf16 product of any number of rows");
  m.def("rows_tile", &rows_tile,
        "bf16 product in tiles: up to 128 rows, more where it is cut over k",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("cols"),
        py::arg("splits"), py::arg("silu") = false);
  m.def("rows_gemm", &rows_gemm, "bf16 product of up to 16 rows");
  m.def("moe_route", &moe_route, "router product and choice");
  m.def("moe_topk", &moe_topk, "softmax routing, top k");
  m.def("moe_choose", &moe_choose,
        "softmax routing of few rows, assignments by expert and the tile list");
  m.def("moe_sort", &moe_sort, "assignments by expert, and the tile list",
        py::arg("experts"), py::arg("E"), py::arg("k"),
        py::arg("weights") = py::none());
  m.def("moe_wide", &moe_wide, "expert products in tiles of up to 320 rows",
        py::arg("down"), py::arg("out"), py::arg("src"), py::arg("w"),
        py::arg("rows"), py::arg("offs"), py::arg("counts"),
        py::arg("s_w") = py::none());
  m.def("moe_sum", &moe_sum, "sum of a row's expert contributions");
  m.def("moe_few", &moe_few, "expert products of few rows an expert",
        py::arg("down"), py::arg("out"), py::arg("src"), py::arg("w"),
        py::arg("rows"), py::arg("tiles"), py::arg("ntiles"), py::arg("offs"),
        py::arg("counts"), py::arg("flat_w") = py::none());
  m.def("moe_tile", &moe_tile, "expert products in 128x128 tiles",
        py::arg("down"), py::arg("out"), py::arg("src"), py::arg("w"),
        py::arg("rows"), py::arg("tiles"), py::arg("ntiles"), py::arg("offs"),
        py::arg("counts"), py::arg("flat_w") = py::none(),
        py::arg("bias") = py::none(), py::arg("act_mode") = 0);
  m.def("wide_rows", &wide_rows,
        "x W^T, or silu(x Wg^T) * (x Wu^T), of many rows (bf16, f32 accum)",
        py::arg("out"), py::arg("x"), py::arg("w"), py::arg("rf"), py::arg("cf"),
        py::arg("silu") = false);
  m.def("wide_parts", &wide_parts, "fp32 parts of a product of many rows",
        py::arg("x"), py::arg("w"), py::arg("splits"), py::arg("rf"), py::arg("cf"));
  m.def("moe_gate_up_silu", &moe_gate_up_silu,
        py::arg("act"), py::arg("x"), py::arg("w"), py::arg("s_tok"),
        py::arg("offs"), py::arg("counts"), py::arg("bias") = py::none(),
        py::arg("act_mode") = 0,
        "grouped MoE gate/up GEMM + SiLU (sorted assignments, sync-free)");
  m.def("moe_down_scale", &moe_down_scale,
        py::arg("contrib"), py::arg("act"), py::arg("w"), py::arg("offs"),
        py::arg("counts"), py::arg("order"), py::arg("flat_w"),
        py::arg("bias") = py::none(),
        py::arg("tiles") = py::none(), py::arg("ntiles") = py::none(),
        "grouped MoE down GEMM + routing-weight scale/scatter");
  m.def("w4_gemm", &w4_gemm,
        "W4A16 GEMM: packed-int4 weights dequantized in-register");
  m.def("w4_parts", &w4_parts,
        "fp32 parts of a W4A16 product that is cut over k, or None");
  m.def("w4_silu", &w4_silu,
        "silu(gate) * up of a W4A16 product, or None");
  m.def("w4_silu_wins",
        [](long M, long N, long K) { return w4_silu_wins(M, N, K); },
        "whether that beats the product and an activation behind it");
  m.def("w4_dequant", &w4_dequant,
        "packed-int4 -> bf16 weight expansion (prefill transient)");
}
