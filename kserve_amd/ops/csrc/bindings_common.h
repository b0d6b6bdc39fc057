// Helpers and the sampling and decode-step wrappers shared by every extension
// module of this package (each links its own copy of sampling.hip and
// decode_step.hip).
#pragma once

#include <torch/extension.h>

#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>

#include <hip/hip_runtime.h>

extern "C" {
hipError_t ks_greedy_sample(void*, const void*, int, int, int, hipStream_t);
hipError_t ks_greedy_advance(void*, const void*, int, int, int, void*, void*, void*, void*,
                             const void*, long, int, int, hipStream_t);
hipError_t ks_gumbel_sample(void*, const void*, const void*, const void*,
                            const void*, int, int, hipStream_t);
hipError_t ks_topk_topp_sample(void*, const void*, const void*, const void*,
                               const void*, const void*, int, int,
                               hipStream_t);
hipError_t ks_unpack_decode_rows(const void*, long, int, int, void*, void*, void*,
                                 void*, void*, void*, long, hipStream_t);
hipError_t ks_advance_decode(const void*, const void*, const void*, void*, void*,
                             void*, void*, void*, void*, long, const void*, long,
                             int, int, int, hipStream_t);
}

namespace {

hipStream_t current_stream() {
  return c10::hip::getCurrentHIPStream().stream();
}

void check_hip(hipError_t err, const char* op) {
  TORCH_CHECK(err == hipSuccess, op, " failed: ", hipGetErrorString(err));
}

#define CHECK_BF16_CONTIG(t)                                       \
  TORCH_CHECK((t).scalar_type() == at::kBFloat16, #t " must be bf16"); \
  TORCH_CHECK((t).is_contiguous(), #t " must be contiguous");      \
  TORCH_CHECK((t).is_cuda(), #t " must be on GPU")

void greedy_sample(at::Tensor& out, at::Tensor& logits) {
  const bool f32 = logits.scalar_type() == at::kFloat;
  if (f32) {
    TORCH_CHECK(logits.is_cuda() && logits.is_contiguous(), "logits [S, V] on GPU");
  } else {
    CHECK_BF16_CONTIG(logits);
  }
  TORCH_CHECK(out.scalar_type() == at::kLong && logits.dim() == 2 &&
                  out.numel() == logits.size(0),
              "out int64 [S]");
  check_hip(ks_greedy_sample(out.data_ptr(), logits.data_ptr(),
                             logits.size(0), logits.size(1), f32 ? 1 : 0,
                             current_stream()),
            "greedy_sample");
}

void gumbel_sample(at::Tensor& out, at::Tensor& logits,
                   at::Tensor& temperatures, at::Tensor& top_k,
                   at::Tensor& seeds) {
  CHECK_BF16_CONTIG(logits);
  TORCH_CHECK(out.scalar_type() == at::kLong, "out int64");
  TORCH_CHECK(temperatures.scalar_type() == at::kFloat, "temps fp32");
  TORCH_CHECK(seeds.scalar_type() == at::kLong, "seeds int64");
  check_hip(ks_gumbel_sample(out.data_ptr(), logits.data_ptr(),
                             temperatures.data_ptr(), top_k.data_ptr(),
                             seeds.data_ptr(), logits.size(0), logits.size(1),
                             current_stream()),
            "gumbel_sample");
}

void topk_topp_sample(at::Tensor& out, at::Tensor& logits,
                      at::Tensor& temperatures, at::Tensor& top_p,
                      at::Tensor& top_k, at::Tensor& seeds) {
  CHECK_BF16_CONTIG(logits);
  TORCH_CHECK(out.scalar_type() == at::kLong, "out int64");
  TORCH_CHECK(temperatures.scalar_type() == at::kFloat, "temps fp32");
  TORCH_CHECK(top_p.scalar_type() == at::kFloat, "top_p fp32");
  TORCH_CHECK(top_k.scalar_type() == at::kInt, "top_k int32");
  TORCH_CHECK(seeds.scalar_type() == at::kLong, "seeds int64");
  check_hip(ks_topk_topp_sample(out.data_ptr(), logits.data_ptr(),
                                temperatures.data_ptr(), top_p.data_ptr(),
                                top_k.data_ptr(), seeds.data_ptr(),
                                logits.size(0), logits.size(1),
                                current_stream()),
            "topk_topp_sample");
}

// operands of a decode step: on device `dev`
#define CHECK_STEP(t, kind, n)                                             \
  TORCH_CHECK((t).device() == dev && (t).scalar_type() == kind && (t).dim() == 1 && \
                  (t).is_contiguous() && (t).numel() >= (n),                  \
              #t ": a dense vector of the rows expected")
#define CHECK_TABLES(t, n)                                                   \
  TORCH_CHECK((t).device() == dev && (t).scalar_type() == at::kInt && (t).dim() == 2 && \
                  (t).size(0) >= (n) && ((t).size(1) < 2 || (t).stride(1) == 1),  \
              #t ": int32 rows expected")

void unpack_decode_rows(at::Tensor& staged, int64_t width, at::Tensor& ids,
                        at::Tensor& positions, at::Tensor& context_lens,
                        at::Tensor& state_slots, at::Tensor& slots,
                        at::Tensor& tables) {
  TORCH_CHECK(ids.is_cuda(), "ids: a GPU tensor expected");
  const c10::Device dev = ids.device();
  const c10::DeviceGuard guard(dev);
  // rows in pinned host memory are read by the kernel itself
  TORCH_CHECK((staged.device() == dev || staged.is_pinned()) &&
                  staged.scalar_type() == at::kInt && staged.dim() == 2 &&
                  staged.is_contiguous(),
              "staged: int32 rows");
  const int64_t rows = staged.size(0);
  CHECK_STEP(ids, at::kLong, rows);
  CHECK_STEP(positions, at::kLong, rows);
  CHECK_STEP(context_lens, at::kInt, rows);
  CHECK_STEP(state_slots, at::kInt, rows);
  CHECK_STEP(slots, at::kInt, rows);
  CHECK_TABLES(tables, rows);
  TORCH_CHECK(width >= 0 && width <= tables.size(1), "table width");
  check_hip(ks_unpack_decode_rows(
                staged.data_ptr(), staged.size(1), (int)rows, (int)width,
                ids.data_ptr(), positions.data_ptr(), context_lens.data_ptr(),
                state_slots.data_ptr(), slots.data_ptr(), tables.data_ptr(),
                std::max<int64_t>(tables.stride(0), tables.size(1)), current_stream()),
            "unpack_decode_rows");
  // pinned rows that are let go of now stay out of use until the kernel has read them,
  // as those of a copy do
  if (!staged.is_cuda()) {
    const at::DataPtr& block = staged.storage().data_ptr();
    at::getHostAllocator(at::kCUDA)->record_event(
        block.get(), block.get_context(),
        c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().unwrap());
  }
}

void advance_decode(at::Tensor& greedy, const c10::optional<at::Tensor>& random,
                    const c10::optional<at::Tensor>& greedy_mask,
                    const c10::optional<at::Tensor>& sampled, at::Tensor& ids,
                    at::Tensor& positions, at::Tensor& context_lens,
                    at::Tensor& slots, const c10::optional<at::Tensor>& seeds,
                    int64_t seed_step, at::Tensor& tables, int64_t block) {
  TORCH_CHECK(greedy.is_cuda(), "greedy: a GPU tensor expected");
  const c10::Device dev = greedy.device();
  const c10::DeviceGuard guard(dev);
  const int64_t rows = greedy.numel();
  CHECK_STEP(greedy, at::kLong, rows);
  CHECK_STEP(ids, at::kLong, rows);
  CHECK_STEP(positions, at::kLong, rows);
  CHECK_STEP(context_lens, at::kInt, rows);
  CHECK_STEP(slots, at::kInt, rows);
  CHECK_TABLES(tables, rows);
  if (random) {
    CHECK_STEP(*random, at::kLong, rows);
    TORCH_CHECK(greedy_mask, "greedy_mask missing");
    CHECK_STEP(*greedy_mask, at::kBool, rows);
  }
  if (sampled) CHECK_STEP(*sampled, at::kLong, rows);
  if (seeds) CHECK_STEP(*seeds, at::kLong, rows);
  check_hip(ks_advance_decode(
                greedy.data_ptr(), random ? random->data_ptr() : nullptr,
                greedy_mask ? greedy_mask->data_ptr() : nullptr,
                sampled ? sampled->data_ptr() : nullptr, ids.data_ptr(),
                positions.data_ptr(), context_lens.data_ptr(), slots.data_ptr(),
                seeds ? seeds->data_ptr() : nullptr, (long)seed_step,
                tables.data_ptr(), tables.stride(0), (int)tables.size(1), (int)block,
                (int)rows, current_stream()),
            "advance_decode");
}

void greedy_advance(at::Tensor& out, at::Tensor& logits, at::Tensor& ids,
                    at::Tensor& positions, at::Tensor& context_lens, at::Tensor& slots,
                    at::Tensor& tables, int64_t block) {
  const bool f32 = logits.scalar_type() == at::kFloat;
  TORCH_CHECK((f32 || logits.scalar_type() == at::kBFloat16) && logits.is_cuda() &&
                  logits.dim() == 2 && logits.is_contiguous() && logits.size(1) > 0,
              "logits bf16 or fp32 [S, V] on GPU");
  const c10::Device dev = logits.device();
  const c10::DeviceGuard guard(dev);
  const int64_t rows = logits.size(0);
  CHECK_STEP(out, at::kLong, rows);
  CHECK_STEP(ids, at::kLong, rows);
  CHECK_STEP(positions, at::kLong, rows);
  CHECK_STEP(context_lens, at::kInt, rows);
  CHECK_STEP(slots, at::kInt, rows);
  CHECK_TABLES(tables, rows);
  check_hip(ks_greedy_advance(out.data_ptr(), logits.data_ptr(), rows, logits.size(1),
                              f32 ? 1 : 0, ids.data_ptr(), positions.data_ptr(),
                              context_lens.data_ptr(), slots.data_ptr(),
                              tables.data_ptr(), tables.stride(0), (int)tables.size(1),
                              (int)block, current_stream()),
            "greedy_advance");
}

void def_sampling(pybind11::module_& m) {
  m.def("unpack_decode_rows", &unpack_decode_rows, "staged decode inputs to buffers");
  m.def("advance_decode", &advance_decode, "the next decode step's inputs");
  m.def("greedy_advance", &greedy_advance, "argmax and the next decode step's inputs");
  m.def("greedy_sample", &greedy_sample, "argmax sampling");
  m.def("gumbel_sample", &gumbel_sample, "Gumbel-max temperature sampling");
  m.def("topk_topp_sample", &topk_topp_sample,
        "fused top-k/top-p + Gumbel-max sampler (radix-histogram select)");
}

}  // namespace
