// Python bindings for the CDNA4 kernels (torch extension, ROCm-native:
// c10::hip stream APIs, no CUDA-compat shims).
#include "bindings_common.h"

// launchers from the .hip translation units
extern "C" {
hipError_t ks_rms_norm(void*, const void*, const void*, float, int, int,
                       hipStream_t);
hipError_t ks_embed_rms_norm(void*, void*, const void*, const void*, const void*, float,
                             int, int, long, hipStream_t);
hipError_t ks_fused_add_rms_norm(void*, void*, const void*, float, int, int,
                                 hipStream_t);
hipError_t ks_silu_and_mul(void*, const void*, int, int, hipStream_t);
hipError_t ks_rotary_embedding(void*, void*, const void*, const void*, int,
                               int, int, int, long, long, hipStream_t);
hipError_t ks_reshape_and_cache(const void*, const void*, void*, void*,
                                const void*, int, int, int, int, long, long,
                                hipStream_t);
hipError_t ks_paged_attention_decode(void*, const void*, const void*,
                                     const void*, const void*, const void*,
                                     float, int, int, int, int, int, int,
                                     long, int, void*, void*, int, int,
                                     hipStream_t);
int ks_paged_decode_splits(int, int, int, int, int);
hipError_t ks_flash_prefill_varlen(void*, const void*, const void*,
                                   const void*, const void*, int, int, int,
                                   int, int, float, long, long, long, int,
                                   int, hipStream_t);
hipError_t ks_context_prefill_varlen(void*, const void*, const void*,
                                     const void*, const void*, const void*,
                                     const void*, int, int, int, int, int,
                                     int, float, long, int, int, long, int,
                                     void*, void*, hipStream_t);
int ks_context_prefill_splits(int, long, int, int, int, int, int);
hipError_t ks_reshape_and_cache_fp8(const void*, const void*, void*, void*,
                                    const void*, int, int, int, int, long,
                                    long, hipStream_t);
hipError_t ks_embed_layer_norm(void*, const void*, const void*, const void*,
                               const void*, const void*, const void*,
                               const void*, const void*, float, int, int, int,
                               int, int, int, void*, hipStream_t);
hipError_t ks_layer_norm(void*, const void*, const void*, const void*, float,
                         int, int, hipStream_t);
hipError_t ks_fused_add_layer_norm(void*, const void*, const void*,
                                   const void*, const void*, float, int, int,
                                   hipStream_t);
hipError_t ks_gelu(void*, const void*, long, hipStream_t);
hipError_t ks_mfma_probe(void*, const void*, const void*, hipStream_t);
hipError_t ks_rope_cache(void*, void*, void*, const void*, int, const void*,
                         const void*, void*, void*, const void*, int, int, int,
                         int, int, int, long, long, long, hipStream_t);
hipError_t ks_add_splits_rms_norm(void*, void*, const void*, const void*, float,
                                  int, int, int, hipStream_t);
int ks_skinny_splits(int, int, int, int);
hipError_t ks_dense_gemm(void*, const void*, const void*, const void*, int, int, int,
                         long, int, int, hipStream_t);
hipError_t ks_skinny_gemm(void*, void*, const void*, const void*, const void*, int, int,
                          int, long, int, int, hipStream_t);
hipError_t ks_streamed_clamped_glu(void*, const void*, const void*, int, int, int, long,
                                   float, float, hipStream_t);
hipError_t ks_gemm8(void*, const void*, const void*, int, int, int, int,
                    hipStream_t);
}

namespace {
// [T, heads, D] where rows may be strided (qkv split views) but the
// (head, dim) block of each row is dense
#define CHECK_KV_CACHE(t)                                               \
  TORCH_CHECK((t).scalar_type() == at::kBFloat16 ||                       \
                  (t).scalar_type() == at::kFloat8_e4m3fn,                \
              #t " must be bf16 or fp8_e4m3");                            \
  TORCH_CHECK((t).is_contiguous(), #t " must be contiguous");             \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU")

#define CHECK_BF16_ROWS(t)                                              \
  TORCH_CHECK((t).scalar_type() == at::kBFloat16, #t " must be bf16");  \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU");                     \
  TORCH_CHECK((t).dim() == 3 && (t).stride(2) == 1 &&                   \
                  (t).stride(1) == (t).size(2),                         \
              #t " inner dims must be dense")

void rms_norm(at::Tensor& out, at::Tensor& input, at::Tensor& weight,
              double eps) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(input);
  CHECK_BF16_CONTIG(weight);
  int hidden = input.size(-1);
  int rows = input.numel() / hidden;
  check_hip(ks_rms_norm(out.data_ptr(), input.data_ptr(), weight.data_ptr(),
                        (float)eps, rows, hidden, current_stream()),
            "rms_norm");
}

void embed_rms_norm(at::Tensor& residual, at::Tensor& out, at::Tensor& table,
                    at::Tensor& ids, at::Tensor& weight, double eps) {
  CHECK_BF16_CONTIG(residual);
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(table);
  CHECK_BF16_CONTIG(weight);
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kLong && ids.is_contiguous(),
              "ids int64");
  TORCH_CHECK(table.dim() == 2 && weight.numel() == table.size(1) && out.dim() == 2 &&
                  out.size(0) == ids.numel() && out.size(1) == table.size(1) &&
                  residual.sizes() == out.sizes(),
              "embed_rms_norm: shape mismatch");
  const c10::Device dev = table.device();
  TORCH_CHECK(residual.device() == dev && out.device() == dev && ids.device() == dev &&
                  weight.device() == dev,
              "operands on different devices");
  const c10::DeviceGuard guard(dev);
  check_hip(ks_embed_rms_norm(residual.data_ptr(), out.data_ptr(), table.data_ptr(),
                              ids.data_ptr(), weight.data_ptr(), (float)eps,
                              (int)out.size(0), (int)out.size(1), table.size(0),
                              current_stream()),
            "embed_rms_norm");
}

void fused_add_rms_norm(at::Tensor& x, at::Tensor& residual, at::Tensor& weight,
                        double eps) {
  CHECK_BF16_CONTIG(x);
  CHECK_BF16_CONTIG(residual);
  int hidden = x.size(-1);
  int rows = x.numel() / hidden;
  check_hip(
      ks_fused_add_rms_norm(x.data_ptr(), residual.data_ptr(),
                            weight.data_ptr(), (float)eps, rows, hidden,
                            current_stream()),
      "fused_add_rms_norm");
}

void silu_and_mul(at::Tensor& out, at::Tensor& input) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(input);
  int d = out.size(-1);
  TORCH_CHECK(input.size(-1) == 2 * d, "input last dim must be 2*out");
  int rows = out.numel() / d;
  check_hip(ks_silu_and_mul(out.data_ptr(), input.data_ptr(), rows, d,
                            current_stream()),
            "silu_and_mul");
}

void rotary_embedding(at::Tensor& positions, at::Tensor& q, at::Tensor& k,
                      at::Tensor& cos_sin_cache) {
  CHECK_BF16_ROWS(q);
  CHECK_BF16_ROWS(k);
  TORCH_CHECK(positions.scalar_type() == at::kLong, "positions must be int64");
  TORCH_CHECK(cos_sin_cache.scalar_type() == at::kFloat,
              "cos_sin_cache must be fp32");
  int T = q.size(0);
  int Hq = q.size(1);
  int Hk = k.size(1);
  int D = q.size(2);
  check_hip(ks_rotary_embedding(q.data_ptr(), k.data_ptr(),
                                positions.data_ptr(), cos_sin_cache.data_ptr(),
                                T, Hq, Hk, D, (long)q.stride(0),
                                (long)k.stride(0), current_stream()),
            "rotary_embedding");
}

void reshape_and_cache(at::Tensor& k, at::Tensor& v, at::Tensor& k_cache,
                       at::Tensor& v_cache, at::Tensor& slot_mapping) {
  CHECK_BF16_ROWS(k);
  CHECK_BF16_ROWS(v);
  CHECK_KV_CACHE(k_cache);
  CHECK_KV_CACHE(v_cache);
  TORCH_CHECK(slot_mapping.scalar_type() == at::kInt, "slot_mapping int32");
  int T = k.size(0);
  int Hkv = k.size(1);
  int D = k.size(2);
  int block_size = k_cache.size(2);
  if (k_cache.scalar_type() == at::kFloat8_e4m3fn) {
    check_hip(ks_reshape_and_cache_fp8(k.data_ptr(), v.data_ptr(),
                                       k_cache.data_ptr(), v_cache.data_ptr(),
                                       slot_mapping.data_ptr(), T, Hkv, D,
                                       block_size, (long)k.stride(0),
                                       (long)v.stride(0), current_stream()),
              "reshape_and_cache_fp8");
    return;
  }
  check_hip(ks_reshape_and_cache(k.data_ptr(), v.data_ptr(),
                                 k_cache.data_ptr(), v_cache.data_ptr(),
                                 slot_mapping.data_ptr(), T, Hkv, D,
                                 block_size, (long)k.stride(0),
                                 (long)v.stride(0), current_stream()),
            "reshape_and_cache");
}

void paged_attention_decode(at::Tensor& out, at::Tensor& q,
                            at::Tensor& k_cache, at::Tensor& v_cache,
                            at::Tensor& block_tables, at::Tensor& context_lens,
                            double scale, int64_t window) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_ROWS(q);
  CHECK_KV_CACHE(k_cache);
  CHECK_KV_CACHE(v_cache);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt, "block_tables int32");
  TORCH_CHECK(context_lens.scalar_type() == at::kInt, "context_lens int32");
  const bool fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
  int S = q.size(0);
  int H = q.size(1);
  int D = q.size(2);
  int Hkv = k_cache.size(1);
  int block_size = k_cache.size(2);
  int max_blocks = block_tables.size(1);
  const int n_splits = ks_paged_decode_splits(S, Hkv, max_blocks, D, fp8);
  at::Tensor part_out, part_ml;
  void *po = nullptr, *pml = nullptr;
  if (n_splits > 1) {
    auto opts = at::TensorOptions().dtype(at::kFloat).device(q.device());
    part_out = at::empty({S, H, n_splits, D}, opts);
    part_ml = at::empty({S, H, n_splits, 2}, opts);
    po = part_out.data_ptr();
    pml = part_ml.data_ptr();
  }
  if (fp8)
    TORCH_CHECK(H / Hkv <= 4 && D == 128,
                "fp8 KV decode supports D=128 and GQA group <= 4");
  check_hip(ks_paged_attention_decode(
                out.data_ptr(), q.data_ptr(), k_cache.data_ptr(),
                v_cache.data_ptr(), block_tables.data_ptr(),
                context_lens.data_ptr(), (float)scale, S, H, Hkv, D,
                max_blocks, block_size, (long)q.stride(0), n_splits, po, pml,
                (int)window, fp8 ? 1 : 0, current_stream()),
            "paged_attention_decode");
}

void flash_prefill_varlen(at::Tensor& out, at::Tensor& q, at::Tensor& k,
                          at::Tensor& v, at::Tensor& cu_seqlens,
                          int64_t max_seqlen, double scale,
                          bool causal = true, int64_t window = 0) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_ROWS(q);
  CHECK_BF16_ROWS(k);
  CHECK_BF16_ROWS(v);
  TORCH_CHECK(cu_seqlens.scalar_type() == at::kInt, "cu_seqlens int32");
  int num_seqs = cu_seqlens.size(0) - 1;
  int Hq = q.size(1);
  int Hkv = k.size(1);
  int D = q.size(2);
  // the kernel's lane offsets are 32 bits wide
  const at::Tensor kk = k.stride(0) < (1L << 26) ? k : k.contiguous();
  const at::Tensor vv = v.stride(0) < (1L << 26) ? v : v.contiguous();
  check_hip(ks_flash_prefill_varlen(out.data_ptr(), q.data_ptr(), kk.data_ptr(),
                                    vv.data_ptr(), cu_seqlens.data_ptr(),
                                    num_seqs, (int)max_seqlen, Hq, Hkv, D,
                                    (float)scale, (long)q.stride(0),
                                    (long)kk.stride(0), (long)vv.stride(0),
                                    causal ? 1 : 0, (int)window,
                                    current_stream()),
            "flash_prefill_varlen");
}

void context_prefill_varlen(at::Tensor& out, at::Tensor& q,
                            at::Tensor& k_cache, at::Tensor& v_cache,
                            at::Tensor& block_tables, at::Tensor& ctx_lens,
                            at::Tensor& cu_seqlens_q, int64_t max_q_len,
                            double scale, int64_t window) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_ROWS(q);
  CHECK_KV_CACHE(k_cache);
  CHECK_KV_CACHE(v_cache);
  TORCH_CHECK(block_tables.scalar_type() == at::kInt, "block_tables int32");
  TORCH_CHECK(block_tables.is_contiguous(), "block_tables contiguous");
  TORCH_CHECK(ctx_lens.scalar_type() == at::kInt, "ctx_lens int32");
  TORCH_CHECK(cu_seqlens_q.scalar_type() == at::kInt, "cu_seqlens_q int32");
  TORCH_CHECK(k_cache.size(2) == 16, "block_size must be 16");
  int num_seqs = cu_seqlens_q.size(0) - 1;
  int Hq = q.size(1);
  int Hkv = k_cache.size(1);
  int D = q.size(2);
  int fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn ? 1 : 0;
  const long rows = (long)q.size(0) * Hq;
  const int n_splits =
      ks_context_prefill_splits(num_seqs, rows, (int)max_q_len, Hq, Hkv,
                                (int)block_tables.size(1), (int)window);
  at::Tensor part_out, part_ml;
  void *po = nullptr, *pml = nullptr;
  if (n_splits > 1) {
    auto opts = at::TensorOptions().dtype(at::kFloat).device(q.device());
    part_out = at::empty({n_splits, rows, D}, opts);
    part_ml = at::empty({n_splits, rows, 2}, opts);
    po = part_out.data_ptr();
    pml = part_ml.data_ptr();
  }
  check_hip(ks_context_prefill_varlen(
                out.data_ptr(), q.data_ptr(), k_cache.data_ptr(),
                v_cache.data_ptr(), block_tables.data_ptr(),
                ctx_lens.data_ptr(), cu_seqlens_q.data_ptr(), num_seqs,
                (int)max_q_len, Hq, Hkv, D, (int)block_tables.size(1),
                (float)scale, (long)q.stride(0), fp8, (int)window, rows, n_splits, po,
                pml, current_stream()),
            "context_prefill_varlen");
}

void embed_layer_norm(at::Tensor& out, at::Tensor& word, at::Tensor& pos_table,
                      at::Tensor& type_table, at::Tensor& ids,
                      const c10::optional<at::Tensor>& types,
                      at::Tensor& cu_seqlens, at::Tensor& weight,
                      at::Tensor& bias, double eps,
                      const c10::optional<at::Tensor>& stats) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(word);
  CHECK_BF16_CONTIG(pos_table);
  CHECK_BF16_CONTIG(type_table);
  CHECK_BF16_CONTIG(weight);
  CHECK_BF16_CONTIG(bias);
  const int64_t hidden = word.size(1), tokens = ids.numel();
  TORCH_CHECK(ids.is_cuda() && ids.scalar_type() == at::kLong &&
                  ids.is_contiguous(),
              "ids int64");
  TORCH_CHECK(cu_seqlens.is_cuda() && cu_seqlens.scalar_type() == at::kInt &&
                  cu_seqlens.is_contiguous() && cu_seqlens.numel() >= 2,
              "cu_seqlens int32 [seqs + 1]");
  if (types.has_value())
    TORCH_CHECK(types->is_cuda() && types->scalar_type() == at::kLong &&
                    types->is_contiguous() && types->numel() == tokens,
                "token types int64 [tokens]");
  TORCH_CHECK(out.dim() == 2 && out.size(0) == tokens && out.size(1) == hidden &&
                  pos_table.size(1) == hidden && type_table.size(1) == hidden &&
                  weight.numel() == hidden && bias.numel() == hidden,
              "embed_layer_norm: shape mismatch");
  const c10::Device dev = word.device();
  if (stats)
    TORCH_CHECK(stats->device() == dev && stats->scalar_type() == at::kLong &&
                    stats->is_contiguous() && stats->numel() == 3,
                "stats int64 [3]");
  TORCH_CHECK(out.device() == dev && pos_table.device() == dev &&
                  type_table.device() == dev && ids.device() == dev &&
                  cu_seqlens.device() == dev && weight.device() == dev &&
                  bias.device() == dev && (!types || types->device() == dev),
              "operands on different devices");
  const c10::DeviceGuard guard(dev);
  check_hip(ks_embed_layer_norm(
                out.data_ptr(), word.data_ptr(), pos_table.data_ptr(),
                type_table.data_ptr(), ids.data_ptr(),
                types.has_value() ? types->data_ptr() : nullptr,
                cu_seqlens.data_ptr(), weight.data_ptr(), bias.data_ptr(),
                (float)eps, (int)tokens, (int)cu_seqlens.numel() - 1, (int)hidden,
                (int)word.size(0), (int)pos_table.size(0),
                (int)type_table.size(0), stats ? stats->data_ptr() : nullptr,
                current_stream()),
            "embed_layer_norm");
}

void layer_norm(at::Tensor& out, at::Tensor& input, at::Tensor& weight,
                at::Tensor& bias, double eps) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(input);
  int hidden = input.size(-1);
  int rows = input.numel() / hidden;
  check_hip(ks_layer_norm(out.data_ptr(), input.data_ptr(), weight.data_ptr(),
                          bias.data_ptr(), (float)eps, rows, hidden,
                          current_stream()),
            "layer_norm");
}

void fused_add_layer_norm(at::Tensor& out, at::Tensor& input,
                          at::Tensor& residual, at::Tensor& weight,
                          at::Tensor& bias, double eps) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(input);
  CHECK_BF16_CONTIG(residual);
  int hidden = input.size(-1);
  int rows = input.numel() / hidden;
  check_hip(ks_fused_add_layer_norm(out.data_ptr(), input.data_ptr(),
                                    residual.data_ptr(), weight.data_ptr(),
                                    bias.data_ptr(), (float)eps, rows, hidden,
                                    current_stream()),
            "fused_add_layer_norm");
}

void gelu(at::Tensor& out, at::Tensor& input) {
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(input);
  check_hip(ks_gelu(out.data_ptr(), input.data_ptr(), input.numel(),
                    current_stream()),
            "gelu");
}

struct SkinnyShape {
  int M, K, N;
  long stride;
};

static SkinnyShape skinny_shape(const at::Tensor& x, const at::Tensor& w, int halves) {
  CHECK_BF16_CONTIG(w);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_cuda() && x.dim() == 2 &&
                  w.dim() == 2 && x.stride(1) == 1,
              "x must be bf16 row-dense");
  const long N = x.size(0), K = x.size(1), M = w.size(0) / halves;
  TORCH_CHECK(w.size(1) == K && w.size(0) == M * halves, "shape mismatch");
  TORCH_CHECK(x.device() == w.device(), "operands on different devices");
  TORCH_CHECK(N >= 1 && N <= 256 && M < (1L << 30) && K < (1L << 30),
              "size out of range");
  return {(int)M, (int)K, (int)N, (long)x.stride(0)};
}

// fp32 sums of the K splits of x @ w^T, [splits][N][M]
static at::Tensor skinny_sums(const at::Tensor& x, const at::Tensor& w) {
  const SkinnyShape z = skinny_shape(x, w, 1);
  const c10::DeviceGuard guard(x.device());
  const int splits = ks_skinny_splits(z.M, z.K, z.N, 0);
  at::Tensor part = at::empty({splits, z.N, z.M}, x.options().dtype(at::kFloat));
  check_hip(ks_skinny_gemm(nullptr, part.data_ptr(), x.data_ptr(), w.data_ptr(), nullptr,
                           z.M, z.K, z.N, z.stride, splits, 0, current_stream()),
            "skinny_gemm");
  return part;
}

static void skinny_product(at::Tensor& out, at::Tensor& x, at::Tensor& w,
                           const c10::optional<at::Tensor>& bias, bool glu) {
  CHECK_BF16_CONTIG(out);
  const SkinnyShape z = skinny_shape(x, w, glu ? 2 : 1);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == z.N && out.size(1) == z.M &&
                  out.device() == x.device(),
              "output shape mismatch");
  if (bias)
    TORCH_CHECK(bias->scalar_type() == at::kBFloat16 && bias->is_contiguous() &&
                    bias->dim() == 1 && bias->size(0) == z.M &&
                    bias->device() == x.device(),
                "bias [M] bf16");
  const c10::DeviceGuard guard(x.device());
  const int splits = ks_skinny_splits(z.M, z.K, z.N, glu);
  at::Tensor part;  // fp32 sums of the K splits
  if (splits > 1)
    part = at::empty({(long)splits * z.N * z.M}, x.options().dtype(at::kFloat));
  check_hip(ks_skinny_gemm(out.data_ptr(), splits > 1 ? part.data_ptr() : nullptr,
                           x.data_ptr(), w.data_ptr(), bias ? bias->data_ptr() : nullptr,
                           z.M, z.K, z.N, z.stride, splits, glu, current_stream()),
            "skinny_gemm");
}

void skinny_gemm(at::Tensor& out, at::Tensor& x, at::Tensor& w,
                 const c10::optional<at::Tensor>& bias) {
  // out [N, M] = x [N, K] @ w [M, K]^T + bias, bf16, N <= 256 (bias: M % 8 == 0)
  skinny_product(out, x, w, bias, false);
}

void skinny_glu(at::Tensor& out, at::Tensor& x, at::Tensor& w) {
  // out [N, M] = silu(x @ w[:M]^T) * (x @ w[M:]^T), bf16, N <= 256
  skinny_product(out, x, w, c10::nullopt, true);
}

void streamed_clamped_glu(at::Tensor& out, at::Tensor& x, at::Tensor& w, double alpha,
                          double limit) {
  // out [N, M] = clamped gate and up of x @ w^T, bf16, N <= 256
  CHECK_BF16_CONTIG(out);
  const SkinnyShape z = skinny_shape(x, w, 2);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == z.N && out.size(1) == z.M &&
                  out.device() == x.device(),
              "output shape mismatch");
  const c10::DeviceGuard guard(x.device());
  check_hip(ks_streamed_clamped_glu(out.data_ptr(), x.data_ptr(), w.data_ptr(), z.M, z.K,
                                    z.N, z.stride, (float)alpha, (float)limit,
                                    current_stream()),
            "streamed_clamped_glu");
}

void dense_gemm(at::Tensor& out, at::Tensor& x, at::Tensor& w,
                const c10::optional<at::Tensor>& bias, bool gelu, int64_t tile) {
  // out [N, M] = act(x [N, K] @ w [M, K]^T + bias), bf16
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(w);
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_cuda() && x.dim() == 2 &&
                  w.dim() == 2 && out.dim() == 2 && x.stride(1) == 1,
              "x must be bf16 row-dense");
  const long N = x.size(0), K = x.size(1), M = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == N && out.size(1) == M, "shape mismatch");
  TORCH_CHECK(x.device() == w.device() && out.device() == x.device(),
              "operands on different devices");
  TORCH_CHECK(N < (1L << 30) && M < (1L << 30) && K < (1L << 30), "size out of range");
  const void* b = nullptr;
  if (bias.has_value()) {
    CHECK_BF16_CONTIG(*bias);
    TORCH_CHECK(bias->numel() == M && bias->device() == x.device(), "bias mismatch");
    b = bias->data_ptr();
  }
  const c10::DeviceGuard guard(x.device());
  check_hip(ks_dense_gemm(out.data_ptr(), x.data_ptr(), w.data_ptr(), b, (int)M, (int)K,
                          (int)N, (long)x.stride(0), gelu ? 1 : 0, (int)tile,
                          current_stream()),
            "dense_gemm");
}

void skinny_add_rms_norm(at::Tensor& out, at::Tensor& residual, at::Tensor& x,
                         at::Tensor& w, at::Tensor& norm_weight, double eps) {
  // residual += x @ w^T; out = RMS norm of residual
  CHECK_BF16_CONTIG(out);
  CHECK_BF16_CONTIG(residual);
  CHECK_BF16_CONTIG(norm_weight);
  const long N = x.size(0), M = w.size(0);
  TORCH_CHECK(out.dim() == 2 && out.size(0) == N && out.size(1) == M &&
                  residual.sizes() == out.sizes() && norm_weight.numel() == M,
              "shape mismatch");
  TORCH_CHECK(x.device() == out.device() && x.device() == residual.device() &&
                  x.device() == norm_weight.device(),
              "operands on different devices");
  const c10::DeviceGuard guard(x.device());
  const at::Tensor part = skinny_sums(x, w);
  check_hip(ks_add_splits_rms_norm(out.data_ptr(), residual.data_ptr(),
                                   part.data_ptr(), norm_weight.data_ptr(),
                                   (float)eps, (int)N, (int)M, (int)part.size(0),
                                   current_stream()),
            "skinny_add_rms_norm");
}

// rotation and scatter, in place or (part) out of the sums of a projection
static void rope_cache_run(at::Tensor& q, at::Tensor& k, at::Tensor& v,
                           const at::Tensor* part, at::Tensor& positions,
                           at::Tensor& cos_sin, at::Tensor& k_cache,
                           at::Tensor& v_cache, at::Tensor& slot_mapping) {
  CHECK_BF16_ROWS(q);
  CHECK_BF16_ROWS(k);
  CHECK_BF16_ROWS(v);
  TORCH_CHECK(positions.scalar_type() == at::kLong, "positions must be int64");
  TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous(),
              "cos_sin_cache must be fp32");
  const int T = q.size(0), Hq = q.size(1), Hk = k.size(1), D = q.size(2);
  TORCH_CHECK(k.size(0) == T && v.sizes() == k.sizes() && k.size(2) == D &&
                  positions.numel() == T && positions.is_contiguous() &&
                  cos_sin.size(-1) == D,
              "rope_and_cache: shape mismatch");
  const c10::Device dev = q.device();
  TORCH_CHECK(k.device() == dev && v.device() == dev && positions.device() == dev &&
                  cos_sin.device() == dev,
              "operands on different devices");
  const c10::DeviceGuard guard(dev);
  const bool cached = k_cache.numel() > 0;
  bool fp8 = false;
  int block = 1;
  if (cached) {
    CHECK_KV_CACHE(k_cache);
    CHECK_KV_CACHE(v_cache);
    TORCH_CHECK(slot_mapping.scalar_type() == at::kInt && slot_mapping.is_contiguous() &&
                    slot_mapping.numel() >= T,
                "slot_mapping int32");
    TORCH_CHECK(k_cache.device() == dev && v_cache.device() == dev &&
                    slot_mapping.device() == dev,
                "pages and slots on another device");
    TORCH_CHECK(k_cache.dim() == 4 && k_cache.size(1) == Hk && k_cache.size(3) == D &&
                    v_cache.sizes() == k_cache.sizes() &&
                    v_cache.scalar_type() == k_cache.scalar_type(),
                "rope_and_cache: page shape mismatch");
    fp8 = k_cache.scalar_type() == at::kFloat8_e4m3fn;
    block = k_cache.size(2);
  }
  check_hip(ks_rope_cache(q.data_ptr(), k.data_ptr(), v.data_ptr(),
                          part ? part->data_ptr() : nullptr,
                          part ? (int)part->size(0) : 0, positions.data_ptr(),
                          cos_sin.data_ptr(), cached ? k_cache.data_ptr() : nullptr,
                          cached ? v_cache.data_ptr() : nullptr,
                          cached ? slot_mapping.data_ptr() : nullptr, T, Hq, Hk, D,
                          block, fp8, (long)q.stride(0), (long)k.stride(0),
                          (long)v.stride(0), current_stream()),
            "rope_and_cache");
}

void rope_and_cache(at::Tensor& positions, at::Tensor& q, at::Tensor& k,
                    at::Tensor& v, at::Tensor& cos_sin, at::Tensor& k_cache,
                    at::Tensor& v_cache, at::Tensor& slot_mapping) {
  rope_cache_run(q, k, v, nullptr, positions, cos_sin, k_cache, v_cache,
                 slot_mapping);
}

void skinny_rope_cache(at::Tensor& q, at::Tensor& k, at::Tensor& v, at::Tensor& x,
                       at::Tensor& w, at::Tensor& positions, at::Tensor& cos_sin,
                       at::Tensor& k_cache, at::Tensor& v_cache,
                       at::Tensor& slot_mapping) {
  // q, k and v (written whole) are the parts of x @ w^T, rotated
  TORCH_CHECK(x.size(0) == q.size(0) &&
                  w.size(0) == (q.size(1) + k.size(1) + v.size(1)) * q.size(2),
              "shape mismatch");
  TORCH_CHECK(x.device() == q.device(), "operands on different devices");
  const c10::DeviceGuard guard(x.device());
  const at::Tensor part = skinny_sums(x, w);
  rope_cache_run(q, k, v, &part, positions, cos_sin, k_cache, v_cache,
                 slot_mapping);
}

void gemm8(at::Tensor& d, at::Tensor& a, at::Tensor& w, int64_t swizzle) {
  // EXPERIMENTAL (see gemm8.hip header): not used by ops.linear dispatch
  CHECK_BF16_CONTIG(d);
  CHECK_BF16_CONTIG(a);
  CHECK_BF16_CONTIG(w);
  int M = a.size(0), K = a.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K && d.size(0) == M && d.size(1) == N,
              "shape mismatch");
  check_hip(ks_gemm8(d.data_ptr(), a.data_ptr(), w.data_ptr(), M, N, K,
                     (int)swizzle, current_stream()),
            "gemm8");
}

void mfma_probe(at::Tensor& c, at::Tensor& a, at::Tensor& b) {
  check_hip(ks_mfma_probe(c.data_ptr(), a.data_ptr(), b.data_ptr(),
                          current_stream()),
            "mfma_probe");
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("rms_norm", &rms_norm, "RMSNorm (bf16, CDNA4)");
  m.def("embed_rms_norm", &embed_rms_norm, "embedding rows and their RMSNorm");
  m.def("fused_add_rms_norm", &fused_add_rms_norm,
        "fused residual-add + RMSNorm, in-place");
  m.def("silu_and_mul", &silu_and_mul, "SwiGLU activation");
  m.def("rotary_embedding", &rotary_embedding, "neox RoPE in-place");
  m.def("reshape_and_cache", &reshape_and_cache, "KV page scatter");
  m.def("paged_attention_decode", &paged_attention_decode,
        "paged decode attention (GQA, split-context)");
  m.def("flash_prefill_varlen", &flash_prefill_varlen,
        "MFMA flash attention (varlen GQA, causal or bidirectional)",
        pybind11::arg("out"), pybind11::arg("q"), pybind11::arg("k"),
        pybind11::arg("v"), pybind11::arg("cu_seqlens"),
        pybind11::arg("max_seqlen"), pybind11::arg("scale"),
        pybind11::arg("causal") = true, pybind11::arg("window") = 0);
  m.def("context_prefill_varlen", &context_prefill_varlen,
        "MFMA prefill attention against the paged KV cache (chunked prefill)");
  namespace py = pybind11;
  m.def("embed_layer_norm", &embed_layer_norm,
        "token + position + type embeddings and their LayerNorm", py::arg("out"),
        py::arg("word"), py::arg("pos_table"), py::arg("type_table"), py::arg("ids"),
        py::arg("types"), py::arg("cu_seqlens"), py::arg("weight"), py::arg("bias"),
        py::arg("eps"), py::arg("stats") = py::none());
  m.def("layer_norm", &layer_norm, "LayerNorm (bf16)");
  m.def("fused_add_layer_norm", &fused_add_layer_norm,
        "residual-add + LayerNorm");
  m.def("gelu", &gelu, "erf GELU");
  def_sampling(m);
  m.def("skinny_gemm", &skinny_gemm, "decode GEMM (N<=256, MFMA streaming)",
        pybind11::arg("out"), pybind11::arg("x"), pybind11::arg("w"),
        pybind11::arg("bias") = pybind11::none());
  m.def("skinny_sums", &skinny_sums, "few-row GEMM as fp32 sums of parts of K");
  m.def("skinny_add_rms_norm", &skinny_add_rms_norm,
        "few-row GEMM into a residual and its RMS norm");
  m.def("rope_and_cache", &rope_and_cache,
        "rotary embedding and K/V scatter in one pass");
  m.def("skinny_rope_cache", &skinny_rope_cache,
        "few-row qkv GEMM, rotary embedding and K/V scatter");
  m.def("skinny_glu", &skinny_glu, "gate|up GEMM (N<=256) with silu(gate) * up");
  m.def("streamed_clamped_glu", &streamed_clamped_glu,
        "gate|up GEMM (N<=256) with the clamped gate");
  m.def("dense_gemm", &dense_gemm, "GEMM with bias and, if asked for, erf GELU",
        pybind11::arg("out"), pybind11::arg("x"), pybind11::arg("w"),
        pybind11::arg("bias"), pybind11::arg("gelu"), pybind11::arg("tile") = -1);
  m.def("gemm8", &gemm8,
        "EXPERIMENTAL 8-phase 256x256 MFMA GEMM");
  m.def("mfma_probe", &mfma_probe, "MFMA layout probe (tests)");
}
