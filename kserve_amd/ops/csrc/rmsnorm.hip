// RMSNorm kernels (bf16, memory-bound).
//
// Replaces the RMSNorm the reference exercises through vLLM/torch
// (SURVEY.md §2.7). Design per CDNA guide Appendix B: vectorized short8
// loads (16 B/lane), one block per token row, grid-stride over rows.
#include "common.h"

namespace {

// Each block handles one row of `hidden` elements; NWAVES=4 (256 threads).
template <bool FUSED_ADD>
__global__ void rms_norm_kernel(
    short* __restrict__ out,          // [rows, hidden] bf16 bits
    short* __restrict__ input,        // [rows, hidden]; FUSED_ADD: in-place normed
    short* __restrict__ residual,     // [rows, hidden] or nullptr
    const short* __restrict__ weight, // [hidden]
    const float eps,
    const int rows,
    const int hidden) {
  constexpr int NWAVES = 4;
  __shared__ float s_partial[NWAVES];
  __shared__ float s_scale;
  const int nvec = hidden >> 3;  // short8 vectors per row

  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    short8_t* row_in = reinterpret_cast<short8_t*>(input) + (size_t)row * nvec;
    short8_t* row_res =
        FUSED_ADD ? reinterpret_cast<short8_t*>(residual) + (size_t)row * nvec
                  : nullptr;
    short8_t* row_out = reinterpret_cast<short8_t*>(out) + (size_t)row * nvec;
    const short8_t* wvec = reinterpret_cast<const short8_t*>(weight);

    float ssq = 0.f;
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = row_in[i];
      float vals[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) vals[j] = bf16_bits_to_float(v[j]);
      if constexpr (FUSED_ADD) {
        short8_t r = row_res[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) vals[j] += bf16_bits_to_float(r[j]);
        short8_t sum;
#pragma unroll
        for (int j = 0; j < 8; ++j) sum[j] = float_to_bf16_bits(vals[j]);
        row_res[i] = sum;  // residual <- x + residual
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ssq += vals[j] * vals[j];
    }
    // block reduce
    int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    ssq = wave_reduce_sum(ssq);
    if (lane == 0) s_partial[wave] = ssq;
    __syncthreads();
    if (threadIdx.x == 0) {
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < NWAVES; ++w) total += s_partial[w];
      s_scale = rsqrtf(total / hidden + eps);
    }
    __syncthreads();
    const float scale = s_scale;

    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      // FUSED_ADD: residual now holds x+residual; re-read it (L2-hot)
      short8_t v = FUSED_ADD ? row_res[i] : row_in[i];
      short8_t w = wvec[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float val = bf16_bits_to_float(v[j]) * scale * bf16_bits_to_float(w[j]);
        o[j] = float_to_bf16_bits(val);
      }
      row_out[i] = o;
    }
    __syncthreads();
  }
}

// residual += sum of the K splits of a projection (fp32, in order), and the
// row's norm, for few rows: a block per row with the row in registers, so the
// splits are read once and the launch that added them is gone. Launch-bound:
// 4.6 us where the two kernels took 4.7 + 4.7 (1 to 77 rows of 4096, 8 splits).
template <int V>
__global__ __launch_bounds__(1024) void add_splits_rms_norm_kernel(
    short* __restrict__ out, short* __restrict__ residual,
    const float* __restrict__ part, const short* __restrict__ weight,
    const float eps, const int rows, const int hidden, const int splits) {
  __shared__ float s_part[16];
  const long row = blockIdx.x, nm = (long)rows * hidden;
  const int step = blockDim.x * 4, at = threadIdx.x * 4;
  float4_t a[V];
  float ssq = 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = at + v * step;
    a[v] = float4_t{0.f, 0.f, 0.f, 0.f};
    if (i >= hidden) continue;
    const float* src = part + row * hidden + i;
    const short4_t r = *reinterpret_cast<const short4_t*>(residual + row * hidden + i);
#pragma unroll 8
    for (int s = 0; s < splits; ++s)
      a[v] += *reinterpret_cast<const float4_t*>(src + s * nm);
    short4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      a[v][j] += bf16_bits_to_float(r[j]);
      o[j] = float_to_bf16_bits(a[v][j]);
      ssq += a[v][j] * a[v][j];
    }
    *reinterpret_cast<short4_t*>(residual + row * hidden + i) = o;
  }
  ssq = wave_reduce_sum(ssq);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = ssq;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) total += s_part[w];
  const float scale = rsqrtf(total / hidden + eps);
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = at + v * step;
    if (i >= hidden) continue;
    const short4_t w = *reinterpret_cast<const short4_t*>(weight + i);
    short4_t o;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      o[j] = float_to_bf16_bits(a[v][j] * scale * bf16_bits_to_float(w[j]));
    *reinterpret_cast<short4_t*>(out + row * hidden + i) = o;
  }
}

// A token's row out of the embedding table and the row's norm: a block per token
// with the row in registers, in the order of sums of the kernel above. A token
// outside the table gets rows of NaN. Few tokens are bound by the launch and the two
// loads that follow each other, many by memory (us, rows of 4096, lookup + norm -> this:
// 1 row 5.5 -> 2.6, 256 5.3 -> 3.4, 2000 12.3 -> 8.6, 8000 41.8 -> 29.5 = 6.6 TB/s).
constexpr int EMBED_NT = 256;

template <int V>
__global__ __launch_bounds__(EMBED_NT) void embed_rms_norm_kernel(
    short* __restrict__ residual, short* __restrict__ out,
    const short* __restrict__ table, const long* __restrict__ ids,
    const short* __restrict__ weight, const float eps, const int hidden,
    const long vocab) {
  __shared__ float s_part[EMBED_NT / 64];
  const long row = blockIdx.x;
  const int nvec = hidden >> 3;
  const long id = ids[row];
  const bool known = id >= 0 && id < vocab;
  const short8_t* src = reinterpret_cast<const short8_t*>(table) + (known ? id : 0) * nvec;
  short8_t x[V], w[V];
  float ssq = 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = threadIdx.x + v * EMBED_NT;
    if (i < nvec) {
      w[v] = reinterpret_cast<const short8_t*>(weight)[i];
      x[v] = src[i];
    }
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = threadIdx.x + v * EMBED_NT;
    if (i >= nvec) continue;
    if (!known) x[v] = (short)0x7fc0;
    reinterpret_cast<short8_t*>(residual)[row * nvec + i] = x[v];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bf16_bits_to_float(x[v][j]);
      ssq += f * f;
    }
  }
  ssq = wave_reduce_sum(ssq);
  if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = ssq;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int k = 0; k < EMBED_NT / 64; ++k) total += s_part[k];
  const float scale = rsqrtf(total / hidden + eps);
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int i = threadIdx.x + v * EMBED_NT;
    if (i >= nvec) continue;
    short8_t o;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = float_to_bf16_bits(bf16_bits_to_float(x[v][j]) * scale *
                                bf16_bits_to_float(w[v][j]));
    if (!known) o = (short)0x7fc0;
    reinterpret_cast<short8_t*>(out)[row * nvec + i] = o;
  }
}

}  // namespace

extern "C" {

// residual <- table[ids], out <- its RMS norm
hipError_t ks_embed_rms_norm(void* residual, void* out, const void* table,
                             const void* ids, const void* weight, float eps, int rows,
                             int hidden, long vocab, hipStream_t stream) {
  if (rows < 0 || vocab < 1 || hidden < 8 || hidden % 8 != 0 || hidden > 16384 ||
      (((uintptr_t)residual | (uintptr_t)out | (uintptr_t)table | (uintptr_t)weight) &
       15) != 0)
    return hipErrorInvalidValue;
  if (rows == 0) return hipSuccess;
#define GO(V)                                                                     \
  hipLaunchKernelGGL((embed_rms_norm_kernel<V>), dim3(rows), dim3(EMBED_NT), 0,   \
                     stream, (short*)residual, (short*)out, (const short*)table,  \
                     (const long*)ids, (const short*)weight, eps, hidden, vocab)
  if (hidden <= 2048) GO(1);
  else if (hidden <= 4096) GO(2);
  else if (hidden <= 8192) GO(4);
  else GO(8);
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

// residual <- residual + sum of splits, out <- its RMS norm
hipError_t ks_add_splits_rms_norm(void* out, void* residual, const void* part,
                                  const void* weight, float eps, int rows,
                                  int hidden, int splits, hipStream_t stream) {
  if (rows < 1 || hidden < 4 || hidden % 4 != 0 || hidden > 16384 || splits < 1 ||
      (((uintptr_t)out | (uintptr_t)residual | (uintptr_t)weight) & 7) != 0 ||
      ((uintptr_t)part & 15) != 0)
    return hipErrorInvalidValue;
  const int vecs = hidden / 4;
  const int threads = vecs >= 1024 ? 1024 : (vecs + 63) / 64 * 64;
  const int v = (vecs + threads - 1) / threads;
#define GO(V)                                                                   \
  hipLaunchKernelGGL((add_splits_rms_norm_kernel<V>), dim3(rows), dim3(threads), \
                     0, stream, (short*)out, (short*)residual,                  \
                     (const float*)part, (const short*)weight, eps, rows,       \
                     hidden, splits)
  if (v == 1) GO(1);
  else if (v == 2) GO(2);
  else GO(4);
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

hipError_t ks_rms_norm(void* out, const void* input, const void* weight,
                       float eps, int rows, int hidden, hipStream_t stream) {
  if (hidden % 8 != 0) return hipErrorInvalidValue;
  int grid = rows < 2048 ? rows : 2048;
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL((rms_norm_kernel<false>), dim3(grid), dim3(256), 0, stream,
                     (short*)out, (short*)input, nullptr, (const short*)weight,
                     eps, rows, hidden);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

// x <- rmsnorm(x + residual), residual <- x + residual (both in-place)
hipError_t ks_fused_add_rms_norm(void* x, void* residual, const void* weight,
                                 float eps, int rows, int hidden,
                                 hipStream_t stream) {
  if (hidden % 8 != 0) return hipErrorInvalidValue;
  int grid = rows < 2048 ? rows : 2048;
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL((rms_norm_kernel<true>), dim3(grid), dim3(256), 0, stream,
                     (short*)x, (short*)x, (short*)residual,
                     (const short*)weight, eps, rows, hidden);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
}
