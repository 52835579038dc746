// Python bindings for the parallax_amd gfx950 kernels (torch extension).

#include <ATen/hip/HIPContext.h>
#include <torch/extension.h>

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <optional>
#include <utility>
#include <vector>

#define CHECK_GPU(x) TORCH_CHECK(x.is_cuda(), #x " must be on GPU")
#define CHECK_CONTIG(x) TORCH_CHECK(x.is_contiguous(), #x " must be contiguous")
#define CHECK_BF16(x) \
  TORCH_CHECK(x.scalar_type() == at::kBFloat16, #x " must be bf16")

extern "C" {
void launch_rmsnorm(void*, void*, const void*, float, int, int, hipStream_t);
void launch_fused_add_rmsnorm(void*, void*, const void*, float, int, int,
                              hipStream_t);
bool norm_linear_takes(int64_t, int64_t, int64_t, bool);
void launch_norm_linear(void*, void*, const void*, const void*, const void*,
                        const void*, const void*, float, int, int, int, int64_t,
                        int64_t, bool, hipStream_t);
void launch_rope(void*, void*, const int*, const float*, int, int, int, int,
                 int, bool, int64_t, int64_t, hipStream_t);
void launch_rope_and_cache(void*, const void*, const void*, void*, void*,
                           const int*, const float*, const int64_t*, int, int,
                           int, int, int, int, bool, bool, float, float,
                           int64_t, int64_t, int64_t, hipStream_t);
void launch_reshape_and_cache(const void*, const void*, void*, void*,
                              const int64_t*, int, int, int, int, hipStream_t);
void launch_mla_reshape_and_cache(const void*, const void*, void*,
                                  const int64_t*, int, int, int, int, bool,
                                  float, hipStream_t);
void launch_mla_rope_and_cache(void*, const void*, const void*, const void*, void*,
                               const int*, const float*, const int64_t*, int, int,
                               int, int, int64_t, int64_t, int64_t, int, float, bool,
                               bool, hipStream_t);
void launch_act_and_mul(void*, const void*, int64_t, int, bool, hipStream_t);
void launch_paged_attention_decode(void*, const void*, const void*, const void*,
                                   const int*, const int*, int, int, int, int,
                                   int, int, int64_t, float, int, float,
                                   const float*, int, int, float*, float*,
                                   hipStream_t, bool*);
struct StackSizes {
  int M, H, Hq, Hk, D, F, max_len;
};
bool decode_stack_takes(const StackSizes*);
int64_t decode_stack_words(const StackSizes*, int (*)[4]);
void launch_decode_stack(const StackSizes*, const void* const*, int, const void*, void*,
                         void*, void*, const int*, const int*, const int*,
                         const int64_t*, const float*, int, int, float, float,
                         hipStream_t);
int paged_decode_runs(int, int, int, int, int);
void launch_paged_decode(void*, const void*, void*, void*, const int*, const int*,
                         int, int, int, int, int, int, int64_t, float, int, float,
                         const float*, int, float*, float*, bool, float, float,
                         const void*, const void*, int64_t, int64_t, const int*,
                         const float*, const int64_t*, hipStream_t, bool*);
void launch_paged_attention_reduce(void*, const float*, const float*, int, int,
                                   int, int, const float*, hipStream_t);
void launch_mla_paged_attention_decode(void*, const void*, const void*,
                                       const void*, const int*, const int*,
                                       int, int, int, int, int, int, float,
                                       int, float*, float*, const int*, int,
                                       bool, hipStream_t, bool*);
int mla_decode_runs(int, int, int);
int mla_prefill_max_portions();
void launch_mla_prefill_paged(void*, const void*, const void*, void*, void*, void*, void*,
                              void*, const void*, const int*, int, int, const void*,
                              const void*, const int*, const int*, int, int, int, int64_t,
                              int64_t, float, hipStream_t);
void launch_mla_prefill_run(void*, float*, const void*, const void*, void*, void*,
                            void*, void*, const void*, const void*, const void*,
                            int, int, int, int, int, int, int64_t, int64_t, float,
                            bool, bool, hipStream_t);
void launch_msa_paged_attention_decode(void*, const void*, const void*,
                                       const void*, const int*, const int*,
                                       const int*, int, int, int, int, int,
                                       int, int, int, int64_t, float,
                                       hipStream_t, bool*);
bool moe_few_takes(int, int, int, int, bool);
void launch_moe_few_gate(void*, const void*, const float*, const void*, const float*,
                         const int64_t*, const float*, const void*, int, int, int, int,
                         int, bool, bool, bool, float, hipStream_t);
void launch_moe_few_down(float*, const void*, const float*, const void*, const float*,
                         const int64_t*, const float*, int, int, int, int, int, bool,
                         bool, hipStream_t);
int moe_tile_rows(int, int, int, bool);
int64_t moe_route_scratch(int, int);
int moe_max_tiles(int, int, int);
void launch_moe_route(int*, void*, int*, int*, const int64_t*, int, int, int, void*,
                      float*, const void*, int, int, hipStream_t);
void launch_moe_gate_up(void*, const void*, const float*, const void*,
                        const float*, const int*, const void*, const int*,
                        const float*, const void*, int, int, int, int, int,
                        bool, bool, bool, float, hipStream_t);
void launch_moe_down(float*, const void*, const float*, const void*,
                     const float*, const int*, const void*, const int*,
                     const float*, int, int, int, int, int, int, int, bool,
                     bool, hipStream_t);
void launch_moe_combine(float*, const float*, const int64_t*, int, int, int,
                        int, int, int, hipStream_t);
int moe_down_cols(int, int);
void launch_dsa_indexer_scores(float*, const void*, const void*, const float*,
                               const int*, const int*, int, int, int, int,
                               int, int, hipStream_t, bool*);
void launch_store_indexer_cache(void*, const void*, const int64_t*, int,
                                int64_t, int, hipStream_t);
void launch_msa_block_scores(float*, const void*, const void*, const int*,
                             const int*, int, int, int, int, int, int, int,
                             int, hipStream_t, bool*);
void launch_msa_topk_tokens(int64_t*, const float*, const int*, int, int, int,
                            int, int, int, int, hipStream_t);
void launch_quantize_fp8_rows(void*, float*, const void*, int, int,
                              hipStream_t);
void launch_sample_gumbel(int64_t*, const float*, const float*,
                          const uint8_t*, uint64_t, int, int, hipStream_t);
void launch_skinny_gemm(void*, const void*, const void*, const void*,
                        const float*, const float*, bool, int, int, int, int64_t,
                        int64_t, int, int64_t, int64_t, bool, hipStream_t, bool*);
int skinny_shared(int, int, int);
bool skinny_pays(int, int, int);
bool skinny_in_pieces(int, int, int, bool, bool);
void skinny_pieces_limits(int*, int64_t*);
void launch_skinny_split(void*, float*, int, const void*, const void*, const void*,
                         const float*, const float*, bool, int, int, int, int64_t,
                         int64_t, bool, hipStream_t);
void launch_mla_absorb(void*, const void*, const void*, int, int, int, int64_t,
                       int64_t, hipStream_t);
int quantize_fp8_tensor_parts(int64_t);
void launch_quantize_fp8_tensor(void*, float*, uint32_t*, const void*, int64_t,
                                bool, int, hipStream_t);
void launch_skinny_norm(void*, void*, uint32_t*, const float*, const void*,
                        const void*, float, int, int, int, int64_t, hipStream_t);
void launch_skinny_add(void*, const float*, const void*, int, int, int, int64_t,
                       hipStream_t);
int silu_and_mul_parts(int64_t, int);
void launch_silu_and_mul_max(void*, uint32_t*, const void*, int64_t, int,
                             hipStream_t);
int prefill_attention_tiles(int, int, int, int);
void launch_prefill_attention(void*, float*, float*, const void*, const void*,
                              const void*, const int*, const int*, const int*,
                              int, int, int, int, int, int, int, int64_t, float,
                              int, float, const float*, int, bool, float, float,
                              hipStream_t, bool*);
}

static hipStream_t cur_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

// [T, H, D] view whose rows may live inside a wider fused tensor (e.g. the QKV
// GEMM output): inner two dims must be dense, the token stride may be larger.
static bool is_fp8(const torch::Tensor& t) {
  return t.scalar_type() == at::kFloat8_e4m3fn;
}

// Kernels that copy memory to LDS directly take 16 bytes from multiples of 16. A
// tensor that begins elsewhere (a view at an odd offset) is copied to one that does.
static torch::Tensor from16(const torch::Tensor& t) {
  return (uintptr_t)t.data_ptr() % 16 ? t.clone() : t;
}

static int64_t row_stride(const torch::Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 3 && t.stride(2) == 1 && t.stride(1) == t.size(2),
              name, " must be [T, H, D] with dense inner dims");
  return t.stride(0);
}

void rmsnorm(torch::Tensor out, torch::Tensor x, torch::Tensor w, double eps) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_BF16(x);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  const int rows = x.numel() / H;
  launch_rmsnorm(out.data_ptr(), x.data_ptr(), w.data_ptr(), (float)eps, rows,
                 H, cur_stream());
}

void fused_add_rmsnorm(torch::Tensor x, torch::Tensor residual, torch::Tensor w,
                       double eps) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_CONTIG(residual);
  CHECK_BF16(x);
  const int H = x.size(-1);
  TORCH_CHECK(H % 8 == 0, "hidden size must be a multiple of 8");
  const int rows = x.numel() / H;
  launch_fused_add_rmsnorm(x.data_ptr(), residual.data_ptr(), w.data_ptr(),
                           (float)eps, rows, H, cur_stream());
}

void rope_inplace(torch::Tensor q, torch::Tensor k, torch::Tensor positions,
                  torch::Tensor cos_sin, bool is_neox) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  TORCH_CHECK(positions.scalar_type() == at::kInt);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat);
  const int T = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k.numel() > 0 ? k.size(1) : 0;
  const int rot = cos_sin.size(-1);
  const int64_t qs = row_stride(q, "q");
  const int64_t ks = Hk ? row_stride(k, "k") : 0;
  launch_rope(q.data_ptr(), Hk ? k.data_ptr() : nullptr,
              positions.data_ptr<int>(), cos_sin.data_ptr<float>(), T, Hq, Hk,
              D, rot, is_neox, qs, ks, cur_stream());
}

void rope_and_cache(torch::Tensor q, torch::Tensor k, torch::Tensor v,
                    torch::Tensor k_cache, torch::Tensor v_cache,
                    torch::Tensor positions, torch::Tensor cos_sin,
                    torch::Tensor slot_mapping, bool is_neox, double k_scale,
                    double v_scale) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  const bool fp8 = is_fp8(k_cache);
  TORCH_CHECK(fp8 || k_cache.scalar_type() == at::kBFloat16,
              "k_cache must be bf16 or fp8_e4m3fn");
  TORCH_CHECK(positions.scalar_type() == at::kInt);
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  const int T = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k.size(1);
  const int BS = k_cache.size(2);
  const int rot = cos_sin.size(-1);
  TORCH_CHECK(rot == D || (rot < D && (D - rot) % 8 == 0));
  launch_rope_and_cache(
      q.data_ptr(), k.data_ptr(), v.data_ptr(), k_cache.data_ptr(),
      v_cache.data_ptr(), positions.data_ptr<int>(), cos_sin.data_ptr<float>(),
      slot_mapping.data_ptr<int64_t>(), T, Hq, Hk, D, rot, BS, is_neox, fp8,
      (float)k_scale, (float)v_scale, row_stride(q, "q"), row_stride(k, "k"),
      row_stride(v, "v"), cur_stream());
}

void reshape_and_cache(torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
                       torch::Tensor v_cache, torch::Tensor slot_mapping) {
  CHECK_GPU(k);
  CHECK_CONTIG(k);
  CHECK_BF16(k_cache);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  const int T = k.size(0);
  const int Hk = k.size(1);
  const int D = k.size(2);
  const int BS = k_cache.size(2);
  TORCH_CHECK((Hk * D) % 8 == 0);
  launch_reshape_and_cache(k.data_ptr(), v.data_ptr(), k_cache.data_ptr(),
                           v_cache.data_ptr(), slot_mapping.data_ptr<int64_t>(),
                           T, Hk, D, BS, cur_stream());
}

void mla_reshape_and_cache(torch::Tensor latent, torch::Tensor k_rope,
                           torch::Tensor cache, torch::Tensor slot_mapping) {
  CHECK_GPU(latent);
  CHECK_CONTIG(latent);
  const int T = latent.size(0);
  const int R = latent.size(-1);
  const int DR = k_rope.size(-1);
  const int BS = cache.size(1);
  TORCH_CHECK(R % 8 == 0 && DR % 8 == 0);
  launch_mla_reshape_and_cache(latent.data_ptr(), k_rope.data_ptr(),
                               cache.data_ptr(),
                               slot_mapping.data_ptr<int64_t>(), T, R, DR, BS,
                               is_fp8(cache), 1.0f, cur_stream());
}

// What mla_rope_and_cache asks of all but kv
static bool mla_rope_takes(const torch::Tensor& q, const torch::Tensor& w,
                           const torch::Tensor& positions,
                           const torch::Tensor& cos_sin, const torch::Tensor& cache,
                           const torch::Tensor& slot_mapping) {
  if (q.dim() != 3 || w.dim() != 1 || cache.dim() != 3 || cos_sin.dim() != 2 ||
      positions.dim() != 1 || slot_mapping.dim() != 1)
    return false;
  const int64_t T = q.size(0), H = q.size(1), DR = q.size(2), R = w.size(0);
  auto at16 = [](const torch::Tensor& t) {
    return (uintptr_t)t.data_ptr() % 16 == 0;
  };
  if (q.scalar_type() != at::kBFloat16 || w.scalar_type() != at::kBFloat16 ||
      (cache.scalar_type() != at::kBFloat16 && !is_fp8(cache)) ||
      cos_sin.scalar_type() != at::kFloat ||
      positions.scalar_type() != at::kInt ||
      slot_mapping.scalar_type() != at::kLong || positions.size(0) != T ||
      slot_mapping.size(0) != T || cos_sin.size(1) != DR || cache.size(2) != R + DR)
    return false;
  // pieces of 16 rotated values, at most a wave of them; vectors of 16 bytes
  return !(T == 0 || T > INT_MAX || H == 0 || R % 8 || DR % 16 || DR > 1024 ||
           H * DR > 1 << 24 || q.stride(2) != 1 || q.stride(1) % 8 ||
           q.stride(0) % 8 || !at16(q) || !at16(w) || !at16(cos_sin) ||
           !at16(cache) || !w.is_contiguous() || !cache.is_contiguous() ||
           !cos_sin.is_contiguous() || !positions.is_contiguous() ||
           !slot_mapping.is_contiguous());
}

// kv: bf16 rows, or (splits > 0) the fp32 parts of their product
static torch::Tensor mla_rope_run(const torch::Tensor& q, const torch::Tensor& kv,
                                  int splits, const torch::Tensor& w, double eps,
                                  const torch::Tensor& positions,
                                  const torch::Tensor& cos_sin,
                                  const torch::Tensor& cache,
                                  const torch::Tensor& slot_mapping, bool neox) {
  const int64_t T = q.size(0), H = q.size(1), DR = q.size(2), R = w.size(0);
  auto out = torch::empty({T, H, DR}, q.options());
  launch_mla_rope_and_cache(
      out.data_ptr(), q.data_ptr(), kv.data_ptr(), w.data_ptr(), cache.data_ptr(),
      positions.data_ptr<int>(), cos_sin.data_ptr<float>(),
      slot_mapping.data_ptr<int64_t>(), T, H, R, DR, q.stride(0), q.stride(1),
      splits > 0 ? 0 : kv.stride(0), splits, (float)eps, neox, is_fp8(cache),
      cur_stream());
  return out;
}

// rotated q [T, H, DR]; kv's normed latent and rotated key go to the cache. None where
// there is no kernel.
std::optional<torch::Tensor> mla_rope_and_cache(
    torch::Tensor q, torch::Tensor kv, torch::Tensor w, double eps,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor cache,
    torch::Tensor slot_mapping, bool neox) {
  CHECK_GPU(q);
  if (!mla_rope_takes(q, w, positions, cos_sin, cache, slot_mapping) ||
      kv.dim() != 2 || kv.scalar_type() != at::kBFloat16 ||
      kv.size(0) != q.size(0) || kv.size(1) != cache.size(2) || kv.stride(1) != 1 ||
      kv.stride(0) % 8 || (uintptr_t)kv.data_ptr() % 16)
    return std::nullopt;
  return mla_rope_run(q, kv, 0, w, eps, positions, cos_sin, cache, slot_mapping, neox);
}

void silu_and_mul(torch::Tensor out, torch::Tensor x) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_BF16(x);
  const int I = out.size(-1);
  TORCH_CHECK(I % 8 == 0);
  launch_act_and_mul(out.data_ptr(), x.data_ptr(), x.numel() / (2 * I), I,
                     false, cur_stream());
}

void gelu_and_mul(torch::Tensor out, torch::Tensor x) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_BF16(x);
  const int I = out.size(-1);
  TORCH_CHECK(I % 8 == 0);
  launch_act_and_mul(out.data_ptr(), x.data_ptr(), x.numel() / (2 * I), I, true,
                     cur_stream());
}

static bool attention_by_valu() {
  static const bool on = std::getenv("PARALLAX_ATTN_VALU") != nullptr;
  return on;
}

void paged_attention_decode(torch::Tensor out, torch::Tensor q,
                            torch::Tensor k_cache, torch::Tensor v_cache,
                            torch::Tensor block_tables, torch::Tensor seq_lens,
                            double scale, int64_t sliding_window,
                            double softcap, torch::Tensor sinks,
                            int64_t max_seq_len, double k_scale,
                            double v_scale) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  const bool kv_fp8 = is_fp8(k_cache);
  TORCH_CHECK(kv_fp8 || k_cache.scalar_type() == at::kBFloat16,
              "k_cache must be bf16 or fp8_e4m3fn");
  TORCH_CHECK(block_tables.scalar_type() == at::kInt);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  const int B = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int max_blocks = block_tables.size(1);
  const int G = Hq / Hk;
  TORCH_CHECK(Hq % Hk == 0 && G <= 16, "GQA group must divide and be <= 16");
  TORCH_CHECK(D == 128 || D == 64, "head_dim must be 64 or 128");
  TORCH_CHECK(BS == 16 || BS == 32 || BS == 64, "block size must be 16/32/64");

  const float* sinks_ptr = nullptr;
  torch::Tensor sinks_f;
  if (sinks.numel() > 0) {
    sinks_f = sinks.to(at::kFloat).contiguous();
    sinks_ptr = sinks_f.data_ptr<float>();
  }

  const bool use_valu = attention_by_valu();
  auto opts = q.options().dtype(at::kFloat);
  torch::Tensor tmp_acc, tmp_ml;
  float *acc_ptr = nullptr, *ml_ptr = nullptr;
  bool launched = false;
  if (!use_valu || kv_fp8) {
    if (B == 0) return;
    k_cache = from16(k_cache);
    v_cache = from16(v_cache);
    // every part of a sequence is named by (run + sequence); see the kernel
    const int runs = paged_decode_runs(B, Hk, D, (int)max_seq_len,
                                       (int)sliding_window);
    if (runs > 0) {
      tmp_acc = torch::empty({(int64_t)runs + B, Hq, D}, opts);
      // of a part each head's maximum and sum; of a sequence its first and last run
      tmp_ml = torch::empty({((int64_t)runs + B) * Hq * 2 + 2 * B}, opts);
      acc_ptr = tmp_acc.data_ptr<float>();
      ml_ptr = tmp_ml.data_ptr<float>();
    }
    launch_paged_decode(
        out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
        block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), B, Hq, Hk, D,
        BS, max_blocks, row_stride(q, "q"), (float)scale, (int)sliding_window,
        (float)softcap, sinks_ptr, runs, acc_ptr, ml_ptr, kv_fp8, (float)k_scale,
        (float)v_scale, nullptr, nullptr, 0, 0, nullptr, nullptr, nullptr,
        cur_stream(), &launched);
    TORCH_CHECK(launched, "no kernel instantiation for D=", D, " BS=", BS,
                " G=", G);
    return;
  }
  // fixed partitions of the context and a reduce kernel
  const int wg_base = B * Hk;
  int part_tokens = 256;
  if (wg_base >= 4096) part_tokens = 2048;
  else if (wg_base >= 1024) part_tokens = 1024;
  else if (wg_base >= 512) part_tokens = 512;
  int num_parts = (int)((max_seq_len + part_tokens - 1) / part_tokens);
  if (num_parts > 128) {
    part_tokens = (int)((max_seq_len + 127) / 128);
    part_tokens = (part_tokens + 127) / 128 * 128;  // chunk-aligned
    num_parts = (int)((max_seq_len + part_tokens - 1) / part_tokens);
  }
  if (num_parts > 1) {
    tmp_acc = torch::empty({B, Hq, num_parts, D}, opts);
    tmp_ml = torch::empty({B, Hq, num_parts, 2}, opts);
    acc_ptr = tmp_acc.data_ptr<float>();
    ml_ptr = tmp_ml.data_ptr<float>();
  }
  launch_paged_attention_decode(
      out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), B, Hq, Hk, D,
      BS, max_blocks, row_stride(q, "q"), (float)scale, (int)sliding_window,
      (float)softcap, sinks_ptr, num_parts, part_tokens, acc_ptr, ml_ptr,
      cur_stream(), &launched);
  TORCH_CHECK(launched, "no kernel instantiation for D=", D, " BS=", BS,
              " G=", G);
  if (num_parts > 1)
    launch_paged_attention_reduce(out.data_ptr(), acc_ptr, ml_ptr, B, Hq, D,
                                  num_parts, sinks_ptr, cur_stream());
}

// rope, the new token into the bf16 cache and decode attention over it; q, k and v are
// left as they are. Every row is its sequence's last token, slot_mapping that token's
// place (or below 0: nothing is stored). None where there is no kernel.
std::optional<torch::Tensor> rope_cache_attention_decode(
    torch::Tensor q, torch::Tensor k, torch::Tensor v, torch::Tensor k_cache,
    torch::Tensor v_cache, torch::Tensor positions, torch::Tensor cos_sin,
    torch::Tensor slot_mapping, torch::Tensor block_tables, torch::Tensor seq_lens,
    double scale, int64_t sliding_window, torch::Tensor sinks, int64_t max_seq_len) {
  CHECK_GPU(q);
  for (const auto* t : {&q, &k, &v})
    if (t->dim() != 3 || t->scalar_type() != at::kBFloat16 || t->stride(2) != 1 ||
        t->stride(1) != t->size(2) || t->stride(0) % 8 ||
        (uintptr_t)t->data_ptr() % 16)
      return std::nullopt;
  if (k_cache.dim() != 4 || v_cache.dim() != 4 || block_tables.dim() != 2 ||
      attention_by_valu())
    return std::nullopt;
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(2), Hk = k.size(1),
                BS = k_cache.size(2);
  for (const auto* t : {&k_cache, &v_cache})
    if (t->scalar_type() != at::kBFloat16 || !t->is_contiguous() ||
        (uintptr_t)t->data_ptr() % 16 || t->size(0) != k_cache.size(0) ||
        t->size(1) != Hk)
      return std::nullopt;
  for (const auto* t : {&positions, &slot_mapping, &seq_lens})
    if (t->dim() != 1 || t->size(0) != B || !t->is_contiguous()) return std::nullopt;
  if (B == 0 || B > 65535 || Hk == 0 || Hq % Hk || Hq / Hk > 15 ||
      (D != 64 && D != 128) || (BS != 16 && BS != 32 && BS != 64) ||
      k.size(0) != B || v.sizes() != k.sizes() || k.size(2) != D ||
      k_cache.size(3) != D || v_cache.size(2) != D || v_cache.size(3) != BS ||
      positions.scalar_type() != at::kInt || seq_lens.scalar_type() != at::kInt ||
      slot_mapping.scalar_type() != at::kLong ||
      block_tables.scalar_type() != at::kInt || block_tables.size(0) != B ||
      !block_tables.is_contiguous() || cos_sin.dim() != 2 || cos_sin.size(1) != D ||
      cos_sin.scalar_type() != at::kFloat || !cos_sin.is_contiguous() ||
      (uintptr_t)cos_sin.data_ptr() % 16 ||
      (sinks.numel() && (sinks.dim() != 1 || sinks.size(0) != Hq ||
                         sinks.scalar_type() != at::kFloat || !sinks.is_contiguous())))
    return std::nullopt;
  auto out = torch::empty({B, Hq, D}, q.options());
  const int runs = paged_decode_runs(B, Hk, D, (int)max_seq_len, (int)sliding_window);
  torch::Tensor acc, ml;
  if (runs > 0) {
    const auto opts = q.options().dtype(at::kFloat);
    acc = torch::empty({runs + B, Hq, D}, opts);
    ml = torch::empty({(runs + B) * Hq * 2 + 2 * B}, opts);
  }
  bool launched = false;
  launch_paged_decode(
      out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), B, Hq, Hk, D, BS,
      block_tables.size(1), q.stride(0), (float)scale, (int)sliding_window, 0.f,
      sinks.numel() ? sinks.data_ptr<float>() : nullptr, runs,
      runs > 0 ? acc.data_ptr<float>() : nullptr,
      runs > 0 ? ml.data_ptr<float>() : nullptr, false, 1.f, 1.f, k.data_ptr(),
      v.data_ptr(), k.stride(0), v.stride(0), positions.data_ptr<int>(),
      cos_sin.data_ptr<float>(), slot_mapping.data_ptr<int64_t>(), cur_stream(),
      &launched);
  TORCH_CHECK(launched, "no kernel instantiation for D=", D, " BS=", BS);
  return out;
}

// Whether decode_stack has a kernel for these sizes.
bool decode_stack_has(int64_t M, int64_t H, int64_t Hq, int64_t Hk, int64_t D, int64_t F,
                      int64_t max_seq_len) {
  for (int64_t v : {M, H, Hq, Hk, D, F, max_seq_len})
    if (v < 1 || v > 1 << 20) return false;
  const StackSizes s{(int)M, (int)H, (int)Hq, (int)Hk, (int)D, (int)F, (int)max_seq_len};
  return decode_stack_takes(&s);
}

// The layers of a Llama-type stack on a decode step of a few rows, in one launch. layers:
// nine tensors each (norm, q/k/v weight, its bias or an empty one, output weight, norm,
// gate and up weight, down weight, K and V cache). Rows are the last tokens of sequences
// of their own, as rope_cache_attention_decode takes them. Returns what the last layer
// adds to the residual stream, and that. None where there is no kernel.
std::optional<std::tuple<torch::Tensor, torch::Tensor>> decode_stack(
    torch::Tensor x, const std::vector<torch::Tensor>& layers, double eps, int64_t Hq,
    int64_t Hk, double scale, torch::Tensor positions, torch::Tensor cos_sin,
    torch::Tensor slot_mapping, torch::Tensor block_tables, torch::Tensor seq_lens,
    int64_t max_seq_len) {
  CHECK_GPU(x);
  constexpr size_t T = 9;  // tensors a layer
  auto plain = [&](const torch::Tensor& t, at::ScalarType type) {
    return t.scalar_type() == type && t.is_contiguous() &&
           (uintptr_t)t.data_ptr() % (type == at::kInt || type == at::kLong ? 4 : 16) == 0 &&
           t.device() == x.device();
  };
  if (layers.empty() || layers.size() % T || x.dim() != 2 ||
      !plain(x, at::kBFloat16) || attention_by_valu())
    return std::nullopt;
  for (const auto& t : layers)
    if (!plain(t, at::kBFloat16)) return std::nullopt;
  const int64_t M = x.size(0), H = x.size(1);
  const auto& k0 = layers[7];
  if (k0.dim() != 4 || layers[6].dim() != 2 || scale <= 0.) return std::nullopt;
  const int64_t NB = k0.size(0), BS = k0.size(2), D = k0.size(3), F = layers[6].size(1),
                N = (Hq + 2 * Hk) * D;
  auto shape = [](const torch::Tensor& t, std::initializer_list<int64_t> s) {
    return t.sizes() == at::IntArrayRef(s);
  };
  if (!decode_stack_has(M, H, Hq, Hk, D, F, max_seq_len)) return std::nullopt;
  for (size_t i = 0; i < layers.size(); i += T) {
    const torch::Tensor* t = &layers[i];
    if (!shape(t[0], {H}) || !shape(t[1], {N, H}) ||
        (t[2].numel() && !shape(t[2], {N})) || !shape(t[3], {H, Hq * D}) ||
        !shape(t[4], {H}) || !shape(t[5], {2 * F, H}) || !shape(t[6], {H, F}) ||
        !shape(t[7], {NB, Hk, BS, D}) || !shape(t[8], {NB, Hk, D, BS}))
      return std::nullopt;
  }
  if ((BS != 16 && BS != 32 && BS != 64) || !plain(positions, at::kInt) ||
      !plain(seq_lens, at::kInt) || !plain(block_tables, at::kInt) ||
      !plain(slot_mapping, at::kLong) || !plain(cos_sin, at::kFloat) ||
      !shape(positions, {M}) || !shape(seq_lens, {M}) || !shape(slot_mapping, {M}) ||
      block_tables.dim() != 2 || block_tables.size(0) != M || cos_sin.dim() != 2 ||
      cos_sin.size(1) != D)
    return std::nullopt;
  const StackSizes sizes{(int)M, (int)H, (int)Hq, (int)Hk, (int)D, (int)F,
                         (int)max_seq_len};
  const int n = (int)(layers.size() / T);
  auto x_out = torch::empty_like(x), res_out = torch::empty_like(x);
  auto work = torch::empty({decode_stack_words(&sizes, nullptr) + (n + 31) / 32 * 16},
                           x.options().dtype(at::kLong));
  std::vector<const void*> pointers(layers.size());
  for (size_t i = 0; i < layers.size(); ++i)
    pointers[i] = layers[i].numel() ? layers[i].data_ptr() : nullptr;
  launch_decode_stack(&sizes, pointers.data(), n, x.data_ptr(), x_out.data_ptr(),
                      res_out.data_ptr(), work.data_ptr(), positions.data_ptr<int>(),
                      seq_lens.data_ptr<int>(), block_tables.data_ptr<int>(),
                      slot_mapping.data_ptr<int64_t>(), cos_sin.data_ptr<float>(),
                      block_tables.size(1), __builtin_ctz((unsigned)BS), (float)eps,
                      (float)scale, cur_stream());
  return std::make_tuple(x_out, res_out);
}

void prefill_attention(torch::Tensor out, torch::Tensor q,
                       torch::Tensor k_cache, torch::Tensor v_cache,
                       torch::Tensor block_tables, torch::Tensor seq_lens,
                       torch::Tensor query_lens, double scale,
                       int64_t sliding_window, double softcap,
                       torch::Tensor sinks, double k_scale, double v_scale) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  const bool kv_fp8 = is_fp8(k_cache);
  TORCH_CHECK(kv_fp8 || k_cache.scalar_type() == at::kBFloat16,
              "k_cache must be bf16 or fp8_e4m3fn");
  TORCH_CHECK(block_tables.scalar_type() == at::kInt);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  TORCH_CHECK(query_lens.scalar_type() == at::kInt &&
              query_lens.is_contiguous());
  const int T = q.size(0);
  const int B = query_lens.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k_cache.size(1);
  const int BS = k_cache.size(2);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(D == 128 || D == 64, "head_dim must be 64 or 128");
  if (T == 0 || B == 0) return;
  k_cache = from16(k_cache);
  v_cache = from16(v_cache);

  const float* sinks_ptr = nullptr;
  torch::Tensor sinks_f;
  if (sinks.numel() > 0) {
    sinks_f = sinks.to(at::kFloat).contiguous();
    sinks_ptr = sinks_f.data_ptr<float>();
  }
  // Short portions on long contexts leave most of the 256 CUs idle: their keys
  // are split over workgroups until two a CU are there, at least 512 keys each
  // (a split writes and reads its fp32 sums once more).
  const int64_t blocks = (int64_t)prefill_attention_tiles(T, B, Hq, Hk) * Hk;
  const int64_t keys = (int64_t)max_blocks * BS;
  int splits = (int)std::max<int64_t>(
      1, std::min<int64_t>({512 / blocks, keys / 512, 64}));
  torch::Tensor tmp_acc, tmp_ml;
  float *acc_ptr = nullptr, *ml_ptr = nullptr;
  if (splits > 1) {
    auto opts = q.options().dtype(at::kFloat);
    tmp_acc = torch::empty({T, Hq, splits, D}, opts);
    tmp_ml = torch::empty({T, Hq, splits, 2}, opts);
    acc_ptr = tmp_acc.data_ptr<float>();
    ml_ptr = tmp_ml.data_ptr<float>();
  }
  bool launched = false;
  launch_prefill_attention(
      out.data_ptr(), acc_ptr, ml_ptr, q.data_ptr(), k_cache.data_ptr(),
      v_cache.data_ptr(), block_tables.data_ptr<int>(),
      seq_lens.data_ptr<int>(), query_lens.data_ptr<int>(), T, B, Hq, Hk, D,
      BS, max_blocks, row_stride(q, "q"), (float)scale, (int)sliding_window,
      (float)softcap, sinks_ptr, splits, kv_fp8, (float)k_scale,
      (float)v_scale, cur_stream(), &launched);
  TORCH_CHECK(launched, "no prefill kernel instantiation for D=", D);
  if (splits > 1)
    launch_paged_attention_reduce(out.data_ptr(), acc_ptr, ml_ptr, T, Hq, D,
                                  splits, sinks_ptr, cur_stream());
}

void mla_paged_attention_decode(torch::Tensor out, torch::Tensor q_latent,
                                torch::Tensor q_pe, torch::Tensor cache,
                                torch::Tensor block_tables,
                                torch::Tensor seq_lens, double scale,
                                int64_t max_seq_len, torch::Tensor topk_indices) {
  CHECK_GPU(q_latent);
  CHECK_CONTIG(q_latent);
  CHECK_CONTIG(q_pe);
  CHECK_BF16(q_latent);
  TORCH_CHECK(cache.scalar_type() == at::kBFloat16 || is_fp8(cache),
              "MLA cache must be bf16 or fp8_e4m3");
  TORCH_CHECK(block_tables.scalar_type() == at::kInt);
  TORCH_CHECK(seq_lens.scalar_type() == at::kInt);
  const int B = q_latent.size(0);
  const int H = q_latent.size(1);
  const int R = q_latent.size(2);
  const int DR = q_pe.size(2);
  const int BS = cache.size(1);
  const int max_blocks = block_tables.size(1);
  TORCH_CHECK(cache.size(2) == R + DR, "cache entry dim mismatch");

  const int* idx_ptr = nullptr;
  int max_topk = 0;
  if (topk_indices.numel() > 0) {
    TORCH_CHECK(topk_indices.scalar_type() == at::kInt &&
                topk_indices.is_contiguous());
    idx_ptr = topk_indices.data_ptr<int>();
    max_topk = topk_indices.size(1);
  }
  // Every part of a sequence is named by (run + sequence); see the kernel.
  const int runs = mla_decode_runs(
      B, H, (int)std::max<int64_t>(max_seq_len, max_topk));
  torch::Tensor tmp_acc, tmp_ml;
  float *acc_ptr = nullptr, *ml_ptr = nullptr;
  if (runs > 0) {
    auto opts = q_latent.options().dtype(at::kFloat);
    tmp_acc = torch::empty({(int64_t)runs + B, H, R}, opts);
    // of a part each head's maximum and sum; of a sequence its first and last run
    tmp_ml = torch::empty({((int64_t)runs + B) * H * 2 + 2 * B}, opts);
    acc_ptr = tmp_acc.data_ptr<float>();
    ml_ptr = tmp_ml.data_ptr<float>();
  }
  if (B == 0) return;
  cache = from16(cache);
  bool launched = false;
  launch_mla_paged_attention_decode(
      out.data_ptr(), q_latent.data_ptr(), q_pe.data_ptr(), cache.data_ptr(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), B, H, R, DR, BS,
      max_blocks, (float)scale, runs, acc_ptr, ml_ptr, idx_ptr, max_topk,
      is_fp8(cache), cur_stream(), &launched);
  TORCH_CHECK(launched, "no MLA kernel for R=", R, " DR=", DR, " BS=", BS);
}

// One request's prompt portion [T, H] over its context rows [L, 512 + 64], the
// portion's own rows last. Returns false where there is no kernel.
bool mla_prefill_attention(torch::Tensor out, torch::Tensor q_nope,
                           torch::Tensor q_pe, torch::Tensor rows,
                           torch::Tensor w_uk, torch::Tensor w_uv, double scale) {
  CHECK_GPU(q_nope);
  const int64_t T = q_nope.size(0), H = q_nope.size(1), L = rows.size(0);
  for (const auto& t : {out, q_nope, q_pe, rows, w_uk, w_uv}) {
    if (t.scalar_type() != at::kBFloat16 || (uintptr_t)t.data_ptr() % 16)
      return false;
  }
  if (q_nope.size(2) != 128 || q_pe.size(2) != 64 || w_uk.size(1) != 128 ||
      w_uv.size(1) != 128 || w_uk.size(2) != 512 || rows.size(1) != 576)
    return false;
  if (q_nope.stride(2) != 1 || q_nope.stride(1) % 8 || q_nope.stride(0) % 8)
    return false;
  if (L < T) return false;
  for (const auto& t : {out, q_pe, rows, w_uk, w_uv})
    if (!t.is_contiguous()) return false;
  TORCH_CHECK(q_pe.size(0) == T && q_pe.size(1) == H && out.size(0) == T &&
              out.size(1) == H && out.size(2) == 128 && w_uk.size(0) == H &&
              w_uv.size(0) == H && w_uv.size(2) == 512);
  if (T == 0 || H == 0) return true;
  // 1 GB of expanded keys and values a run
  const int64_t run = std::max<int64_t>(128, ((1 << 20) / H) & ~127);
  const int64_t cap = (std::min(L, run) + 127) & ~127;
  auto kv = torch::empty({4, H * cap * 128}, q_nope.options());
  torch::Tensor state;
  if (L > run)
    state = torch::empty({T, H, 130}, q_nope.options().dtype(at::kFloat));
  uint16_t* p = (uint16_t*)kv.data_ptr();
  const size_t part = (size_t)H * cap * 128;
  for (int64_t k0 = 0; k0 < L; k0 += run) {
    const int64_t n = std::min(run, L - k0);
    launch_mla_prefill_run(
        out.data_ptr(), L > run ? state.data_ptr<float>() : nullptr,
        q_nope.data_ptr(), q_pe.data_ptr(), p, p + part, p + 2 * part,
        p + 3 * part, (const uint16_t*)rows.data_ptr() + k0 * 576,
        w_uk.data_ptr(), w_uv.data_ptr(), T, H, n, cap, L - T, k0,
        q_nope.stride(0), q_nope.stride(1), (float)scale, k0 == 0, k0 + n == L,
        cur_stream());
  }
  return true;
}

// Portions of requests over their contexts in cache [NB, BS, 576]: lens (rows, context
// rows with them) of each, whose rows lie one behind the other in q and out and whose
// pages are the rows of block_tables. False where there is no kernel.
bool mla_prefill_paged(torch::Tensor out, torch::Tensor q_nope, torch::Tensor q_pe,
                       torch::Tensor cache, torch::Tensor block_tables,
                       std::vector<std::pair<int64_t, int64_t>> lens, torch::Tensor w_uk,
                       torch::Tensor w_uv, double scale) {
  CHECK_GPU(q_nope);
  const int64_t T = q_nope.size(0), H = q_nope.size(1);
  for (const auto& t : {out, q_nope, q_pe, cache, w_uk, w_uv}) {
    if (t.dim() != 3 || t.scalar_type() != at::kBFloat16 ||
        (uintptr_t)t.data_ptr() % 16 || t.device() != q_nope.device())
      return false;
  }
  const int64_t BS = cache.size(1);
  if (q_nope.size(2) != 128 || q_pe.size(2) != 64 || w_uk.size(1) != 128 ||
      w_uv.size(1) != 128 || w_uk.size(2) != 512 || cache.size(2) != 576 || BS < 1 ||
      BS > 1 << 20 || (BS & (BS - 1)))
    return false;
  if (q_nope.stride(2) != 1 || q_nope.stride(1) % 8 || q_nope.stride(0) % 8)
    return false;
  for (const auto& t : {out, q_pe, cache, w_uk, w_uv, block_tables})
    if (!t.is_contiguous()) return false;
  if (block_tables.dim() != 2 || block_tables.scalar_type() != at::kInt ||
      block_tables.device() != q_nope.device() ||
      (int64_t)lens.size() > block_tables.size(0))
    return false;
  TORCH_CHECK(q_pe.size(0) == T && q_pe.size(1) == H && out.size(0) == T &&
              out.size(1) == H && out.size(2) == 128 && w_uk.size(0) == H &&
              w_uv.size(0) == H && w_uv.size(2) == 512);
  if (H == 0) return true;
  // 1 GB of expanded keys and values a pair of launches; a longer context goes by runs.
  // Short prompts together take it too: 16 of 512 rows, 128 heads all of it, where one
  // request at a time takes 67 MB.
  const int64_t run = std::max<int64_t>(128, ((1 << 20) / H) & ~127);
  struct Request { int64_t rows, context, first, seq; };
  std::vector<Request> all;
  int64_t at = 0;
  for (size_t i = 0; i < lens.size(); ++i) {
    const auto [rows, context] = lens[i];
    if (rows < 0 || context < rows || context > run ||
        (context + BS - 1) / BS > block_tables.size(1))
      return false;
    if (rows > 0) all.push_back({rows, context, at, (int64_t)i});
    at += rows;
  }
  if (at > T) return false;
  std::stable_sort(all.begin(), all.end(), [](const Request& a, const Request& b) {
    return a.context < b.context;
  });
  const size_t most = mla_prefill_max_portions();
  for (size_t i = 0; i < all.size();) {
    std::vector<int> sizes, starts;
    int64_t cap = 0;
    size_t j = i;
    for (; j < all.size() && j - i < most; ++j) {
      const int64_t more = (all[j].context + 127) & ~127;
      if (j > i && cap + more > run) break;
      cap += more;
      sizes.insert(sizes.end(), {(int)all[j].rows, (int)all[j].context});
      starts.insert(starts.end(), {(int)all[j].first, (int)all[j].seq});
    }
    const int64_t part = H * cap * 128;
    auto kv = torch::empty({4 * part + cap * 64}, q_nope.options());
    uint16_t* p = (uint16_t*)kv.data_ptr();
    launch_mla_prefill_paged(
        out.data_ptr(), q_nope.data_ptr(), q_pe.data_ptr(), p, p + part, p + 2 * part,
        p + 3 * part, p + 4 * part, cache.data_ptr(), block_tables.data_ptr<int>(),
        block_tables.size(1), __builtin_ctzll(BS), w_uk.data_ptr(), w_uv.data_ptr(),
        sizes.data(), starts.data(), (int)(j - i), H, cap, q_nope.stride(0),
        q_nope.stride(1), (float)scale, cur_stream());
    i = j;
  }
  return true;
}

// Routed experts of x [T, H]: bf16, or fp8 (W8A8) with w_gu_scale / w_down_scale
// given. Returns fp32 [T, H].
static torch::Tensor moe_layer(torch::Tensor x, torch::Tensor w_gu,
                               torch::Tensor w_gu_scale, torch::Tensor w_down,
                               torch::Tensor w_down_scale,
                               torch::Tensor topk_ids, torch::Tensor topk_w,
                               bool gelu, double limit, torch::Tensor bias_gu,
                               bool weight_on_input, bool fp8) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_BF16(x);
  CHECK_CONTIG(w_gu);
  CHECK_CONTIG(w_down);
  TORCH_CHECK(topk_ids.dim() == 2 && topk_ids.is_contiguous() &&
              topk_ids.scalar_type() == at::kLong);
  TORCH_CHECK(topk_w.is_contiguous() && topk_w.scalar_type() == at::kFloat &&
              topk_w.numel() == topk_ids.numel());
  const int T = x.size(0);
  const int k = topk_ids.size(1);
  const int E = w_gu.size(0);
  const int I = w_gu.size(1) / 2;
  const int H = w_gu.size(2);
  const int n = T * k;
  TORCH_CHECK(topk_ids.size(0) == T && x.size(1) == H &&
              w_down.size(0) == E && w_down.size(1) == H &&
              w_down.size(2) == I, "MoE operand shapes do not match");
  TORCH_CHECK(H % 32 == 0 && I % (fp8 ? 64 : 32) == 0,
              "MoE dims must be multiples of 32, fp8 I of 64 (H=", H, " I=", I,
              ")");
  TORCH_CHECK(bias_gu.numel() == 0 ||
              (bias_gu.scalar_type() == at::kBFloat16 &&
               bias_gu.is_contiguous() &&
               bias_gu.numel() == (int64_t)E * 2 * I));
  auto fopts = x.options().dtype(at::kFloat);
  auto bopts = x.options().dtype(at::kByte);
  if (n == 0) return torch::zeros({T, H}, fopts);
  x = from16(x);
  w_gu = from16(w_gu);
  w_down = from16(w_down);
  auto stream = cur_stream();

  const int64_t* ids = topk_ids.data_ptr<int64_t>();
  const float* wts = topk_w.data_ptr<float>();
  const bool few = moe_few_takes(n, E, H, I, fp8);
  const int tm = moe_tile_rows(n, E, I, fp8);
  const int max_tiles = moe_max_tiles(n, E, tm);
  // tiles (16 bytes each) first, then their number, the order, the counts
  torch::Tensor ws;
  int *tiles = nullptr, *n_tiles = nullptr, *perm = nullptr;
  if (!few) {
    ws = torch::empty({4 * (int64_t)max_tiles + 4 + n + moe_route_scratch(n, E)},
                      x.options().dtype(at::kInt));
    tiles = ws.data_ptr<int>();
    n_tiles = tiles + 4 * (int64_t)max_tiles;
    perm = n_tiles + 4;
  }

  torch::Tensor xq, xs, hq, hs;
  const void* xp = x.data_ptr();
  if (fp8) {
    xq = torch::empty({T, H}, bopts);
    xs = torch::empty({T}, fopts);
    if (few)
      launch_quantize_fp8_rows(xq.data_ptr(), xs.data_ptr<float>(), xp, T, H,
                               stream);
  }
  if (!few)
    launch_moe_route(perm, tiles, n_tiles, perm + n, ids, n, E, tm,
                     fp8 ? xq.data_ptr() : nullptr, fp8 ? xs.data_ptr<float>() : nullptr,
                     xp, T, H, stream);
  if (fp8) xp = xq.data_ptr();
  torch::Tensor h = torch::empty({n, I}, x.options());
  const float* gus = fp8 ? w_gu_scale.data_ptr<float>() : nullptr;
  const float* ds = fp8 ? w_down_scale.data_ptr<float>() : nullptr;
  const void* bias = bias_gu.numel() ? bias_gu.data_ptr() : nullptr;
  if (few)
    launch_moe_few_gate(h.data_ptr(), xp, fp8 ? xs.data_ptr<float>() : nullptr,
                        w_gu.data_ptr(), gus, ids, wts, bias, n, k, E, H, I, fp8,
                        weight_on_input, gelu, (float)limit, stream);
  else
    launch_moe_gate_up(h.data_ptr(), xp, fp8 ? xs.data_ptr<float>() : nullptr,
                       w_gu.data_ptr(), gus, perm, tiles, n_tiles, wts, bias, k, H, I,
                       max_tiles, tm, fp8, weight_on_input, gelu, (float)limit, stream);
  const void* hp = h.data_ptr();
  if (fp8) {
    hq = torch::empty({n, I}, bopts);
    hs = torch::empty({n}, fopts);
    launch_quantize_fp8_rows(hq.data_ptr(), hs.data_ptr<float>(), hp, n, I,
                             stream);
    hp = hq.data_ptr();
  }
  torch::Tensor out = torch::empty({T, H}, fopts);
  if (few) {
    launch_moe_few_down(out.data_ptr<float>(), hp, fp8 ? hs.data_ptr<float>() : nullptr,
                        w_down.data_ptr(), ds, ids, wts, n, k, E, H, I, fp8,
                        weight_on_input, stream);
    return out;
  }
  const int slab = moe_down_cols(n, H);
  torch::Tensor y = torch::empty({n, slab}, fopts);
  for (int first = 0; first < H; first += slab) {
    const int cols = std::min(slab, H - first);
    launch_moe_down(y.data_ptr<float>(), hp,
                    fp8 ? hs.data_ptr<float>() : nullptr, w_down.data_ptr(), ds, perm,
                    tiles, n_tiles, wts, k, H, I, first, cols, max_tiles, tm, fp8,
                    weight_on_input, stream);
    launch_moe_combine(out.data_ptr<float>(), y.data_ptr<float>(), ids, T, k, E,
                       H, first, cols, stream);
  }
  return out;
}

torch::Tensor moe_forward(torch::Tensor x, torch::Tensor w_gu,
                          torch::Tensor w_down, torch::Tensor topk_ids,
                          torch::Tensor topk_w, bool gelu, double limit,
                          torch::Tensor bias_gu, bool weight_on_input) {
  CHECK_BF16(w_gu);
  CHECK_BF16(w_down);
  return moe_layer(x, w_gu, {}, w_down, {}, topk_ids, topk_w, gelu, limit,
                   bias_gu, weight_on_input, false);
}

torch::Tensor moe_forward_fp8(torch::Tensor x, torch::Tensor w_gu,
                              torch::Tensor w_gu_scale, torch::Tensor w_down,
                              torch::Tensor w_down_scale,
                              torch::Tensor topk_ids, torch::Tensor topk_w,
                              bool gelu, double limit) {
  TORCH_CHECK(is_fp8(w_gu) && is_fp8(w_down));
  TORCH_CHECK(w_gu_scale.scalar_type() == at::kFloat &&
              w_down_scale.scalar_type() == at::kFloat &&
              w_gu_scale.is_contiguous() && w_down_scale.is_contiguous());
  return moe_layer(x, w_gu, w_gu_scale, w_down, w_down_scale, topk_ids, topk_w,
                   gelu, limit, x.new_empty({0}), false, true);
}

torch::Tensor dsa_indexer_scores(torch::Tensor q_index,
                                 torch::Tensor index_cache,
                                 torch::Tensor head_weights,
                                 torch::Tensor block_tables,
                                 torch::Tensor seq_lens, int64_t max_ctx) {
  CHECK_GPU(q_index);
  CHECK_BF16(q_index);
  CHECK_BF16(index_cache);
  TORCH_CHECK(index_cache.dim() == 3, "index cache must be [NB, BS, Di]");
  TORCH_CHECK(head_weights.scalar_type() == at::kFloat);
  const int B = q_index.size(0);
  const int Hi = q_index.size(1);
  const int Di = q_index.size(2);
  const int BS = index_cache.size(1);
  auto scores = torch::empty(
      {B, max_ctx}, q_index.options().dtype(at::kFloat));
  bool launched = false;
  launch_dsa_indexer_scores(
      scores.data_ptr<float>(), q_index.contiguous().data_ptr(),
      index_cache.data_ptr(), head_weights.contiguous().data_ptr<float>(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(), B, Hi, Di, BS,
      block_tables.size(1), (int)max_ctx, cur_stream(), &launched);
  TORCH_CHECK(launched, "no dsa_indexer kernel for Hi=", Hi, " Di=", Di);
  return scores;
}

void store_indexer_cache(torch::Tensor index_keys, torch::Tensor index_cache,
                         torch::Tensor slot_mapping, int64_t trash_slot) {
  CHECK_GPU(index_keys);
  CHECK_BF16(index_keys);
  CHECK_BF16(index_cache);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kLong);
  const int T = index_keys.size(0);
  const int DI = index_keys.size(-1);
  TORCH_CHECK(DI % 8 == 0);
  launch_store_indexer_cache(index_cache.data_ptr(),
                             index_keys.contiguous().data_ptr(),
                             slot_mapping.data_ptr<int64_t>(), T, trash_slot,
                             DI, cur_stream());
}

torch::Tensor msa_block_scores(torch::Tensor q, torch::Tensor k_cache,
                               torch::Tensor block_tables,
                               torch::Tensor seq_lens, int64_t sparse_block,
                               int64_t max_sparse_blocks) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  CHECK_BF16(k_cache);
  const int B = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k_cache.size(1);
  const int BS = k_cache.size(2);
  auto out = torch::empty(
      {B, max_sparse_blocks}, q.options().dtype(at::kFloat));
  bool launched = false;
  launch_msa_block_scores(out.data_ptr<float>(), q.contiguous().data_ptr(),
                          k_cache.data_ptr(), block_tables.data_ptr<int>(),
                          seq_lens.data_ptr<int>(), B, Hq, Hk, D, BS,
                          block_tables.size(1), (int)sparse_block,
                          (int)max_sparse_blocks, cur_stream(), &launched);
  TORCH_CHECK(launched, "no msa_block_scores kernel for D=", D);
  return out;
}

torch::Tensor msa_topk_tokens(torch::Tensor block_scores,
                              torch::Tensor seq_lens, int64_t sparse_block,
                              int64_t topk_blocks, int64_t init_blocks,
                              int64_t local_blocks, int64_t max_positions) {
  CHECK_GPU(block_scores);
  TORCH_CHECK(block_scores.scalar_type() == at::kFloat);
  const int B = block_scores.size(0);
  auto out = torch::empty(
      {B, max_positions}, block_scores.options().dtype(at::kLong));
  launch_msa_topk_tokens(out.data_ptr<int64_t>(),
                         block_scores.contiguous().data_ptr<float>(),
                         seq_lens.data_ptr<int>(), B, (int)sparse_block,
                         block_scores.size(1), (int)topk_blocks,
                         (int)init_blocks, (int)local_blocks,
                         (int)max_positions, cur_stream());
  return out;
}

torch::Tensor sample_gumbel(torch::Tensor logits, torch::Tensor inv_temp,
                            torch::Tensor greedy, int64_t seed) {
  CHECK_GPU(logits);
  CHECK_CONTIG(logits);
  TORCH_CHECK(logits.scalar_type() == at::kFloat, "logits must be fp32");
  TORCH_CHECK(inv_temp.scalar_type() == at::kFloat);
  TORCH_CHECK(greedy.scalar_type() == at::kByte);
  const int B = logits.size(0);
  const int V = logits.size(1);
  auto out = torch::empty({B}, logits.options().dtype(at::kLong));
  launch_sample_gumbel(out.data_ptr<int64_t>(), logits.data_ptr<float>(),
                       inv_temp.contiguous().data_ptr<float>(),
                       greedy.contiguous().data_ptr<uint8_t>(),
                       (uint64_t)seed, B, V, cur_stream());
  return out;
}

// c = x . w^T (+ bias): bf16, or fp8 with the two scales given; gated: c = silu(first
// half of the columns) * second half. False where there is no kernel; c is allocated
// where it is not given, once there is one.
static bool skinny_run(torch::Tensor& c, torch::Tensor x, torch::Tensor w,
                       torch::Tensor bias, torch::Tensor x_scale,
                       torch::Tensor w_scale, bool gated) {
  CHECK_GPU(x);
  const bool fp8 = x_scale.numel() > 0;
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1) &&
              x.stride(1) == 1);
  CHECK_CONTIG(w);
  if (c.defined()) {
    TORCH_CHECK(c.dim() == 2 && c.stride(1) == 1 && c.size(0) == x.size(0) &&
                c.size(1) * (gated ? 2 : 1) == w.size(0));
    CHECK_BF16(c);
    if ((uintptr_t)c.data_ptr() % 8 || c.stride(0) % 4) return false;
  }
  if (fp8) {
    TORCH_CHECK(is_fp8(x) && is_fp8(w) &&
                x_scale.scalar_type() == at::kFloat &&
                w_scale.scalar_type() == at::kFloat);
    if (w_scale.numel() != 1) return false;
  } else {
    CHECK_BF16(x);
    CHECK_BF16(w);
  }
  CHECK_BF16(bias);
  if (bias.numel() && (bias.dim() != 1 || bias.numel() != w.size(0) ||
                       !bias.is_contiguous()))
    return false;
  if (w.numel() == 0) return false;
  const int64_t es = x.element_size();
  // the kernels place rows of x by 32-bit offsets
  if ((x.size(0) - 1) * x.stride(0) * es + 128 > UINT32_MAX) return false;
  if ((uintptr_t)x.data_ptr() % 16 || (uintptr_t)w.data_ptr() % 16 ||
      x.stride(0) * es % 16)
    return false;
  const int M = x.size(0), N = w.size(0), row_bytes = x.size(1) * es;
  const void* b = bias.numel() ? bias.data_ptr() : nullptr;
  const float* xs = fp8 ? x_scale.data_ptr<float>() : nullptr;
  const float* ws = fp8 ? w_scale.data_ptr<float>() : nullptr;
  // gated: halves as silu_and_mul takes them, offsets of 32 bits from row 0 on
  if (gated && (N % 16 || (int64_t)N * row_bytes > UINT32_MAX)) return false;
  const int splits = x.is_contiguous() && skinny_in_pieces(M, N, row_bytes, gated, b != nullptr)
                         ? 0 : skinny_shared(M, N, row_bytes);
  if (splits < 0) return false;
  if (!c.defined())
    c = torch::empty({M, gated ? N / 2 : N}, x.options().dtype(at::kBFloat16));
  if (splits > 0) {
    torch::Tensor part;
    if (splits > 1)
      part = torch::empty({splits, M, N}, x.options().dtype(at::kFloat));
    launch_skinny_split(c.data_ptr(), splits > 1 ? part.data_ptr<float>() : nullptr,
                        splits, x.data_ptr(), w.data_ptr(), b, xs, ws, fp8, M, N,
                        row_bytes, x.stride(0) * es, c.stride(0), gated,
                        cur_stream());
    return true;
  }
  bool launched = false;
  launch_skinny_gemm(c.data_ptr(), x.data_ptr(), w.data_ptr(), b, xs, ws, fp8, M, N,
                     row_bytes, x.stride(0) * es, c.stride(0), 1, 0, 0, gated,
                     cur_stream(), &launched);
  return launched;
}

bool skinny_gemm(torch::Tensor c, torch::Tensor x, torch::Tensor w,
                 torch::Tensor bias, torch::Tensor x_scale, torch::Tensor w_scale,
                 bool gated) {
  return skinny_run(c, x, w, bias, x_scale, w_scale, gated);
}

// (f(rms_norm(x + res)) . w^T + bias, x + res) of few rows: bf16; without a norm (empty)
// or res (empty) neither is there. None where there is no kernel.
std::optional<std::tuple<torch::Tensor, torch::Tensor>> norm_linear(
    torch::Tensor x, torch::Tensor res, torch::Tensor norm, double eps,
    torch::Tensor w, torch::Tensor bias, bool gated) {
  CHECK_GPU(x);
  CHECK_BF16(x);
  CHECK_BF16(w);
  CHECK_BF16(res);
  CHECK_BF16(norm);
  CHECK_BF16(bias);
  TORCH_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(1));
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  const bool has_norm = norm.numel() > 0, has_res = res.numel() > 0;
  auto rows16 = [](const torch::Tensor& t) {
    return (uintptr_t)t.data_ptr() % 16 == 0 && t.stride(1) == 1 &&
           t.stride(0) % 8 == 0;
  };
  if (!norm_linear_takes(M, N, K, has_norm) || !rows16(x) || !rows16(w) ||
      !w.is_contiguous() || (gated && N % 2))
    return std::nullopt;
  if (has_res && (!has_norm || res.dim() != 2 || res.size(0) != M ||
                  res.size(1) != K || !rows16(res)))
    return std::nullopt;
  if (has_norm && (norm.dim() != 1 || norm.size(0) != K || !norm.is_contiguous() ||
                   (uintptr_t)norm.data_ptr() % 16))
    return std::nullopt;
  if (bias.numel() && (bias.dim() != 1 || bias.size(0) != N || !bias.is_contiguous()))
    return std::nullopt;
  auto c = torch::empty({M, gated ? N / 2 : N}, x.options());
  auto sum = has_res ? torch::empty({M, K}, x.options()) : x;
  launch_norm_linear(c.data_ptr(), sum.data_ptr(), x.data_ptr(),
                     has_res ? res.data_ptr() : nullptr,
                     has_norm ? norm.data_ptr() : nullptr, w.data_ptr(),
                     bias.numel() ? bias.data_ptr() : nullptr, (float)eps, M, N, K,
                     x.stride(0), has_res ? res.stride(0) : 0, gated, cur_stream());
  return std::make_tuple(c, sum);
}

// skinny_gemm with the result allocated; None where there is no kernel, or the library
// is faster
std::optional<torch::Tensor> few_rows(torch::Tensor x, torch::Tensor w,
                                      torch::Tensor bias, torch::Tensor x_scale,
                                      torch::Tensor w_scale, bool gated) {
  torch::Tensor c;
  // gated: halves as silu_and_mul takes them, for any number of rows
  if (x_scale.numel() == 0 && x.dim() == 2 && w.dim() == 2 &&
      !(gated && w.size(0) % 16) &&
      norm_linear_takes(x.size(0), w.size(0), x.size(1), false)) {
    const auto none = w.new_empty({0});
    auto r = norm_linear(x, none, none, 0., w, bias, gated);
    if (r) return std::get<0>(*r);
  }
  const int64_t row_bytes = x.size(1) * x.element_size();
  if (!gated && !skinny_pays(x.size(0), w.size(0), row_bytes) &&
      !(x.is_contiguous() &&
        skinny_in_pieces(x.size(0), w.size(0), row_bytes, false, bias.numel() > 0)))
    return std::nullopt;
  if (!skinny_run(c, x, w, bias, x_scale, w_scale, gated)) return std::nullopt;
  return c;
}

// x quantised per tensor: (fp8 values, scale [1])
std::tuple<torch::Tensor, torch::Tensor> quantize_fp8_tensor(torch::Tensor x) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 || x.scalar_type() == at::kFloat);
  TORCH_CHECK(x.numel() > 0, "quantize_fp8_tensor: empty input");
  auto q = torch::empty(x.sizes(), x.options().dtype(at::kFloat8_e4m3fn));
  const int64_t n = x.numel();
  auto scale = torch::empty({1}, x.options().dtype(at::kFloat));
  auto part = torch::empty({quantize_fp8_tensor_parts(n)},
                           x.options().dtype(at::kInt));
  launch_quantize_fp8_tensor(q.data_ptr(), scale.data_ptr<float>(),
                             (uint32_t*)part.data_ptr(), x.data_ptr(), n,
                             x.scalar_type() == at::kBFloat16, 0, cur_stream());
  return {q, scale};
}

// fp8 values of bf16 x and their scale, from its parts' largest magnitudes
static std::tuple<torch::Tensor, torch::Tensor> quantize_by_parts(
    const torch::Tensor& x, const torch::Tensor& part) {
  auto q = torch::empty(x.sizes(), x.options().dtype(at::kFloat8_e4m3fn));
  auto scale = torch::empty({1}, x.options().dtype(at::kFloat));
  launch_quantize_fp8_tensor(q.data_ptr(), scale.data_ptr<float>(),
                             (uint32_t*)part.data_ptr(), x.data_ptr(), x.numel(), true,
                             (int)part.numel(), cur_stream());
  return {q, scale};
}

// silu(first half) * second half of bf16 rows, as fp8 values and their scale
std::tuple<torch::Tensor, torch::Tensor> silu_and_mul_fp8(torch::Tensor x) {
  CHECK_GPU(x);
  CHECK_CONTIG(x);
  CHECK_BF16(x);
  TORCH_CHECK(x.dim() == 2 && x.numel() > 0 && x.size(1) % 16 == 0);
  const int64_t T = x.size(0), I = x.size(1) / 2;
  auto h = torch::empty({T, I}, x.options());
  auto part = torch::empty({silu_and_mul_parts(T, I)}, x.options().dtype(at::kInt));
  launch_silu_and_mul_max(h.data_ptr(), (uint32_t*)part.data_ptr(), x.data_ptr(), T, I,
                          cur_stream());
  return quantize_by_parts(h, part);
}

// parts that linear() of few rows adds up in a launch of their own, 0: none
int64_t product_parts(int64_t M, int64_t N, int64_t row_bytes) {
  if (M < 1 || M > 128 || N < 1 || N > 8192 || row_bytes < 1 || row_bytes > INT_MAX ||
      !skinny_pays(M, N, row_bytes))
    return 0;
  const int splits = skinny_shared(M, N, row_bytes);
  return splits > 1 ? splits : 0;
}

// The parts [splits, M, N] of x . w^T of few rows, for a launch that adds them up to rows
// beside those of residual. fp8 w takes its own scale, and bf16 x or fp8 x with x_scale.
// None where linear() has no parts, and for operands that no such launch takes.
static std::optional<torch::Tensor> product_in_parts(
    const torch::Tensor& x, const torch::Tensor& x_scale, const torch::Tensor& w,
    const torch::Tensor& w_scale, const torch::Tensor& residual) {
  const bool fp8 = is_fp8(w), has_res = residual.numel() > 0, ready = x_scale.numel() > 0;
  auto rows16 = [](const torch::Tensor& t) {
    return (uintptr_t)t.data_ptr() % 16 == 0 && t.stride(1) == 1;
  };
  if (x.dim() != 2 || w.dim() != 2 || x.numel() == 0 || w.numel() == 0 ||
      x.size(1) != w.size(1) || !w.is_contiguous() ||
      (!fp8 && w.scalar_type() != at::kBFloat16) ||
      (ready ? !fp8 || !is_fp8(x) || x_scale.numel() != 1 ||
                   x_scale.scalar_type() != at::kFloat || !rows16(x)
             : x.scalar_type() != at::kBFloat16))
    return std::nullopt;
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  if (M > 128 || N > 8192 || N % 8 || K > INT_MAX / 2 || !rows16(w)) return std::nullopt;
  if (has_res && (residual.dim() != 2 || residual.size(0) != M ||
                  residual.size(1) != N || !rows16(residual) ||
                  residual.stride(0) % 8 ||
                  residual.scalar_type() != at::kBFloat16))
    return std::nullopt;
  if (fp8 ? w_scale.numel() != 1 || w_scale.scalar_type() != at::kFloat ||
                !x.is_contiguous()
          : !rows16(x) || x.stride(0) % 8)
    return std::nullopt;
  const int64_t row_bytes = K * w.element_size();
  if ((M - 1) * (fp8 ? K : x.stride(0) * 2) + 128 > UINT32_MAX) return std::nullopt;
  const int splits = product_parts(M, N, row_bytes);
  if (splits <= 1) return std::nullopt;
  torch::Tensor scale = x_scale, xq = x;
  if (fp8 && !ready) std::tie(xq, scale) = quantize_fp8_tensor(x);
  auto part = torch::empty({splits, M, N}, x.options().dtype(at::kFloat));
  launch_skinny_split(nullptr, part.data_ptr<float>(), splits, xq.data_ptr(),
                      w.data_ptr(), nullptr, fp8 ? scale.data_ptr<float>() : nullptr,
                      fp8 ? w_scale.data_ptr<float>() : nullptr, fp8, M, N, row_bytes,
                      xq.stride(0) * xq.element_size(), 0, false, cur_stream());
  return part;
}

// rms_norm(x . w^T + residual) of few rows whose product is split over K: (the normed
// rows, as fp8 values with their scale where quantize is set, else bf16 and an empty
// scale; product + residual, empty without one). None where there is no kernel or
// linear() has none.
std::optional<std::tuple<torch::Tensor, torch::Tensor, torch::Tensor>> linear_norm(
    torch::Tensor x, torch::Tensor x_scale, torch::Tensor w, torch::Tensor w_scale,
    torch::Tensor residual, torch::Tensor norm, double eps, bool quantize) {
  CHECK_GPU(x);
  if (w.dim() != 2 || norm.dim() != 1 || norm.scalar_type() != at::kBFloat16 ||
      norm.size(0) != w.size(0) || !norm.is_contiguous() ||
      (uintptr_t)norm.data_ptr() % 16)
    return std::nullopt;
  const auto part = product_in_parts(x, x_scale, w, w_scale, residual);
  if (!part) return std::nullopt;
  const bool has_res = residual.numel() > 0;
  const int splits = part->size(0), M = part->size(1), N = part->size(2);
  const auto bf16 = x.options().dtype(at::kBFloat16);
  auto out = torch::empty({M, N}, bf16);
  auto sum = torch::empty({has_res ? M : 0, N}, bf16);
  torch::Tensor top;
  if (quantize) top = torch::empty({M}, x.options().dtype(at::kInt));
  launch_skinny_norm(out.data_ptr(), has_res ? sum.data_ptr() : nullptr,
                     quantize ? (uint32_t*)top.data_ptr() : nullptr,
                     part->data_ptr<float>(), has_res ? residual.data_ptr() : nullptr,
                     norm.data_ptr(), (float)eps, splits, M, N,
                     has_res ? residual.stride(0) : 0, cur_stream());
  if (!quantize)
    return std::make_tuple(out, x.new_empty({0}, at::kFloat), sum);
  auto [q, scale] = quantize_by_parts(out, top);
  return std::make_tuple(q, scale, sum);
}

// x . w^T + residual of few rows whose product is split over K; None as linear_norm.
std::optional<torch::Tensor> linear_add(torch::Tensor x, torch::Tensor x_scale,
                                        torch::Tensor w, torch::Tensor w_scale,
                                        torch::Tensor residual) {
  CHECK_GPU(x);
  if (residual.numel() == 0) return std::nullopt;
  const auto part = product_in_parts(x, x_scale, w, w_scale, residual);
  if (!part) return std::nullopt;
  const int splits = part->size(0), M = part->size(1), N = part->size(2);
  auto out = torch::empty({M, N}, residual.options());
  launch_skinny_add(out.data_ptr(), part->data_ptr<float>(), residual.data_ptr(), splits,
                    M, N, residual.stride(0), cur_stream());
  return out;
}

// mla_rope_and_cache of kv = x . kv_w^T, whose parts its launch adds up. None where
// linear() has none for that product, and where mla_rope_and_cache has no kernel.
std::optional<torch::Tensor> linear_mla_rope_and_cache(
    torch::Tensor x, torch::Tensor kv_w, torch::Tensor q, torch::Tensor w, double eps,
    torch::Tensor positions, torch::Tensor cos_sin, torch::Tensor cache,
    torch::Tensor slot_mapping, bool neox) {
  CHECK_GPU(x);
  if (!mla_rope_takes(q, w, positions, cos_sin, cache, slot_mapping) ||
      x.dim() != 2 || kv_w.dim() != 2 || x.scalar_type() != at::kBFloat16 ||
      kv_w.scalar_type() != at::kBFloat16 || x.size(0) != q.size(0) ||
      x.size(1) != kv_w.size(1) || kv_w.size(0) != cache.size(2) ||
      !kv_w.is_contiguous() || (uintptr_t)kv_w.data_ptr() % 16 ||
      (uintptr_t)x.data_ptr() % 16 || x.stride(1) != 1 || x.stride(0) % 8)
    return std::nullopt;
  const int64_t M = x.size(0), K = x.size(1), N = kv_w.size(0);
  if (M > 128 || K == 0 || K > INT_MAX / 2 ||
      (M - 1) * x.stride(0) * 2 + 128 > UINT32_MAX)
    return std::nullopt;
  const int splits = product_parts(M, N, K * 2);
  if (splits <= 1) return std::nullopt;
  auto part = torch::empty({splits, M, N}, x.options().dtype(at::kFloat));
  launch_skinny_split(nullptr, part.data_ptr<float>(), splits, x.data_ptr(),
                      kv_w.data_ptr(), nullptr, nullptr, nullptr, false, M, N, K * 2,
                      x.stride(0) * 2, 0, false, cur_stream());
  return mla_rope_run(q, part, splits, w, eps, positions, cos_sin, cache, slot_mapping,
                      neox);
}

static bool rows16(const torch::Tensor& t) {
  return t.scalar_type() == at::kBFloat16 && (uintptr_t)t.data_ptr() % 16 == 0 &&
         t.stride(2) == 1 && t.stride(1) % 8 == 0 && t.stride(0) % 8 == 0;
}

// MLA's per-head products with bf16 results [B, H, R] and [B, H, dv]; false where
// there is no kernel.
bool mla_absorb(torch::Tensor out, torch::Tensor q, torch::Tensor w) {
  CHECK_GPU(q);
  const int64_t B = q.size(0), H = q.size(1), R = w.size(2);
  if (!rows16(q) || !rows16(w) || !w.is_contiguous() || q.size(2) != 128 ||
      R % 128)
    return false;
  CHECK_CONTIG(out);
  CHECK_BF16(out);
  TORCH_CHECK(w.size(0) == H && w.size(1) == 128 && out.size(0) == B &&
              out.size(1) == H && out.size(2) == R);
  if (out.numel() == 0) return true;
  launch_mla_absorb(out.data_ptr(), q.data_ptr(), w.data_ptr(), B, H, R,
                    q.stride(0), q.stride(1), cur_stream());
  return true;
}

bool mla_project(torch::Tensor out, torch::Tensor x, torch::Tensor w) {
  CHECK_GPU(x);
  const int64_t B = x.size(0), H = x.size(1), N = w.size(1), K = w.size(2);
  if (!rows16(x) || !rows16(w) || !w.is_contiguous() || K % 64 || N % 64)
    return false;
  // rows go 32 at a time, placed by 32-bit offsets
  if (31 * x.stride(0) * 2 + 128 > UINT32_MAX) return false;
  CHECK_CONTIG(out);
  CHECK_BF16(out);
  TORCH_CHECK(w.size(0) == H && x.size(2) == K && out.size(0) == B &&
              out.size(1) == H && out.size(2) == N);
  if (out.numel() == 0) return true;
  bool launched = false;
  launch_skinny_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), nullptr, nullptr,
                     nullptr, false, B, N, K * 2, x.stride(0) * 2, out.stride(0),
                     H, x.stride(1) * 2, out.stride(1), false, cur_stream(),
                     &launched);
  return launched;
}

void msa_paged_attention_decode(torch::Tensor out, torch::Tensor q,
                                torch::Tensor k_cache, torch::Tensor v_cache,
                                torch::Tensor block_tables,
                                torch::Tensor seq_lens,
                                torch::Tensor token_positions, double scale) {
  CHECK_GPU(q);
  CHECK_BF16(q);
  CHECK_BF16(k_cache);
  TORCH_CHECK(token_positions.scalar_type() == at::kInt &&
              token_positions.is_contiguous());
  const int B = q.size(0);
  const int Hq = q.size(1);
  const int D = q.size(2);
  const int Hk = k_cache.size(1);
  const int BS = k_cache.size(2);
  // token_positions: [B, P] shared across kv heads, or [B, Hk, P] per head
  const int pos_heads = token_positions.dim() == 3 ? token_positions.size(1) : 1;
  if (pos_heads > 1)
    TORCH_CHECK(pos_heads == Hk, "positions head dim must equal Hk");
  bool launched = false;
  launch_msa_paged_attention_decode(
      out.data_ptr(), q.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
      block_tables.data_ptr<int>(), seq_lens.data_ptr<int>(),
      token_positions.data_ptr<int>(), token_positions.size(-1), pos_heads, B,
      Hq, Hk, D, BS, block_tables.size(1), row_stride(q, "q"), (float)scale,
      cur_stream(), &launched);
  TORCH_CHECK(launched, "no MSA kernel for D=", D, " BS=", BS, " G=", Hq / Hk);
}

torch::Tensor lt_linear(torch::Tensor x, torch::Tensor w);  // lt_gemm.cpp
torch::Tensor lt_linear_fp8(torch::Tensor x_q, torch::Tensor w_q,
                            torch::Tensor x_scale, torch::Tensor w_scale);

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("lt_linear_fp8", &lt_linear_fp8,
        "fp8-E4M3 W8A8 y = (xq*sx) @ (wq*sw)^T (bf16 out)");
  m.def("lt_linear", &lt_linear,
        "tuned hipBLASLt y = x @ w^T (bf16, fp32 accum)");
  m.def("msa_paged_attention_decode", &msa_paged_attention_decode);
  m.def("skinny_gemm", &skinny_gemm);
  m.def("few_rows", &few_rows);
  m.def("norm_linear", &norm_linear);
  m.def("skinny_pieces_limits", [] {
    int rows;
    int64_t bytes;
    skinny_pieces_limits(&rows, &bytes);
    return std::make_tuple(rows, bytes);
  });
  m.def("moe_few_takes", &moe_few_takes);
  m.def("decode_stack", &decode_stack);
  m.def("decode_stack_has", &decode_stack_has);
  m.def("quantize_fp8_tensor", &quantize_fp8_tensor);
  m.def("silu_and_mul_fp8", &silu_and_mul_fp8);
  m.def("linear_add", &linear_add);
  m.def("linear_norm", &linear_norm);
  m.def("product_parts", &product_parts);
  m.def("mla_absorb", &mla_absorb);
  m.def("mla_project", &mla_project);
  m.def("sample_gumbel", &sample_gumbel);
  m.def("moe_forward", &moe_forward);
  m.def("moe_forward_fp8", &moe_forward_fp8);
  m.def("dsa_indexer_scores", &dsa_indexer_scores);
  m.def("store_indexer_cache", &store_indexer_cache);
  m.def("msa_block_scores", &msa_block_scores);
  m.def("msa_topk_tokens", &msa_topk_tokens);
  m.def("mla_paged_attention_decode", &mla_paged_attention_decode);
  m.def("mla_prefill_attention", &mla_prefill_attention);
  m.def("mla_prefill_paged", &mla_prefill_paged);
  m.def("prefill_attention", &prefill_attention);
  m.def("rmsnorm", &rmsnorm);
  m.def("fused_add_rmsnorm", &fused_add_rmsnorm);
  m.def("rope_inplace", &rope_inplace);
  m.def("rope_and_cache", &rope_and_cache);
  m.def("reshape_and_cache", &reshape_and_cache);
  m.def("mla_reshape_and_cache", &mla_reshape_and_cache);
  m.def("mla_rope_and_cache", &mla_rope_and_cache);
  m.def("linear_mla_rope_and_cache", &linear_mla_rope_and_cache);
  m.def("silu_and_mul", &silu_and_mul);
  m.def("gelu_and_mul", &gelu_and_mul);
  m.def("paged_attention_decode", &paged_attention_decode);
  m.def("rope_cache_attention_decode", &rope_cache_attention_decode);
}
