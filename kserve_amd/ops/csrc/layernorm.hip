// LayerNorm (+ optional fused residual add) and GELU — the encoder-path
// (BERT-class) elementwise ops. Memory-bound; vectorized short8 per CDNA
// guide Appendix B.
#include "common.h"

#include <climits>

namespace {

template <bool FUSED_ADD>
__global__ void layer_norm_kernel(
    short* __restrict__ out,           // [rows, hidden]
    const short* __restrict__ input,   // [rows, hidden]
    const short* __restrict__ residual,  // [rows, hidden] or nullptr
    const short* __restrict__ weight,  // [hidden]
    const short* __restrict__ bias,    // [hidden]
    const float eps, const int rows, const int hidden) {
  constexpr int NWAVES = 4;
  __shared__ float s_sum[NWAVES];
  __shared__ float s_sq[NWAVES];
  __shared__ float s_mean, s_rstd;
  const int nvec = hidden >> 3;

  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const short8_t* rin = reinterpret_cast<const short8_t*>(input) + (size_t)row * nvec;
    const short8_t* rres =
        FUSED_ADD ? reinterpret_cast<const short8_t*>(residual) + (size_t)row * nvec
                  : nullptr;
    short8_t* rout = reinterpret_cast<short8_t*>(out) + (size_t)row * nvec;
    const short8_t* wv = reinterpret_cast<const short8_t*>(weight);
    const short8_t* bv = reinterpret_cast<const short8_t*>(bias);

    float sum = 0.f, sq = 0.f;
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = rin[i];
      short8_t r;
      if constexpr (FUSED_ADD) r = rres[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf16_bits_to_float(v[j]);
        if constexpr (FUSED_ADD) f += bf16_bits_to_float(r[j]);
        sum += f;
        sq += f * f;
      }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    sum = wave_reduce_sum(sum);
    sq = wave_reduce_sum(sq);
    if (lane == 0) {
      s_sum[wave] = sum;
      s_sq[wave] = sq;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      float ts = 0.f, tq = 0.f;
#pragma unroll
      for (int w = 0; w < NWAVES; ++w) {
        ts += s_sum[w];
        tq += s_sq[w];
      }
      const float mean = ts / hidden;
      const float var = tq / hidden - mean * mean;
      s_mean = mean;
      s_rstd = rsqrtf(var + eps);
    }
    __syncthreads();
    const float mean = s_mean, rstd = s_rstd;
    for (int i = threadIdx.x; i < nvec; i += blockDim.x) {
      short8_t v = rin[i];
      short8_t r;
      if constexpr (FUSED_ADD) r = rres[i];
      short8_t w = wv[i];
      short8_t b = bv[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float f = bf16_bits_to_float(v[j]);
        if constexpr (FUSED_ADD) f += bf16_bits_to_float(r[j]);
        f = (f - mean) * rstd * bf16_bits_to_float(w[j]) +
            bf16_bits_to_float(b[j]);
        o[j] = float_to_bf16_bits(f);
      }
      rout[i] = o;
    }
    __syncthreads();
  }
}

// Rows of up to 2048: a wave per row with the row in registers, read once, no
// barrier, and the variance from the centred values. Bound by memory: 6400 rows
// of 768 with the residual take 9.2 us, 10.1 us with a block per row (of whose
// 256 threads 96 had a vector).
template <bool FUSED_ADD, int V>
__global__ __launch_bounds__(256) void layer_norm_wave_kernel(
    short* __restrict__ out, const short* __restrict__ input,
    const short* __restrict__ residual, const short* __restrict__ weight,
    const short* __restrict__ bias, const float eps, const int rows,
    const int hidden) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= rows) return;
  const int nvec = hidden >> 3;
  const long at = (long)row * nvec;
  float x[V][8];
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const int i = lane + 64 * u;
    if (i < nvec) {
      const short8_t a = reinterpret_cast<const short8_t*>(input)[at + i];
      short8_t r;
      if constexpr (FUSED_ADD) r = reinterpret_cast<const short8_t*>(residual)[at + i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[u][j] = bf16_bits_to_float(a[j]);
        if constexpr (FUSED_ADD) x[u][j] += bf16_bits_to_float(r[j]);
        sum += x[u][j];
      }
    }
  }
  const float mean = wave_reduce_sum(sum) / hidden;
  float sq = 0.f;
#pragma unroll
  for (int u = 0; u < V; ++u)
    if (lane + 64 * u < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sq += (x[u][j] - mean) * (x[u][j] - mean);
    }
  const float rstd = rsqrtf(wave_reduce_sum(sq) / hidden + eps);
#pragma unroll
  for (int u = 0; u < V; ++u) {
    const int i = lane + 64 * u;
    if (i < nvec) {
      const short8_t w = reinterpret_cast<const short8_t*>(weight)[i];
      const short8_t b = reinterpret_cast<const short8_t*>(bias)[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = float_to_bf16_bits((x[u][j] - mean) * rstd * bf16_bits_to_float(w[j]) +
                                  bf16_bits_to_float(b[j]));
      reinterpret_cast<short8_t*>(out)[at + i] = o;
    }
  }
}

template <bool FUSED_ADD>
hipError_t launch_layer_norm(void* out, const void* input, const void* residual,
                             const void* weight, const void* bias, float eps,
                             int rows, int hidden, hipStream_t stream) {
  if (hidden % 8 != 0) return hipErrorInvalidValue;
  if (rows < 1) return hipSuccess;
#define LN_ARGS                                                           \
  (short*)out, (const short*)input, (const short*)residual,               \
      (const short*)weight, (const short*)bias, eps, rows, hidden
#define LN_WAVE(V)                                                        \
  hipLaunchKernelGGL((layer_norm_wave_kernel<FUSED_ADD, V>),              \
                     dim3((rows + 3) / 4), dim3(256), 0, stream, LN_ARGS)
  if (hidden <= 512) LN_WAVE(1);
  else if (hidden <= 1024) LN_WAVE(2);
  else if (hidden <= 2048) LN_WAVE(4);
  else
    hipLaunchKernelGGL((layer_norm_kernel<FUSED_ADD>),
                       dim3(rows < 2048 ? rows : 2048), dim3(256), 0, stream,
                       LN_ARGS);
#undef LN_WAVE
#undef LN_ARGS
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

__global__ void gelu_kernel(short* __restrict__ out,
                            const short* __restrict__ input, const long nvec) {
  const short8_t* in = reinterpret_cast<const short8_t*>(input);
  short8_t* ov = reinterpret_cast<short8_t*>(out);
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < nvec;
       i += (long)gridDim.x * blockDim.x) {
    short8_t v = in[i];
    short8_t o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float x = bf16_bits_to_float(v[j]);
      // erf-based gelu (matches torch default / BERT)
      o[j] = float_to_bf16_bits(0.5f * x * (1.f + erff(x * 0.70710678f)));
    }
    ov[i] = o;
  }
}

// Sum of a token's word, position and type rows, then LayerNorm, a wave per
// token with the row in registers (hidden <= 2048). The position is the
// token's place in its sequence, found in cu_seqlens (relative to its first
// entry). Negative ids count from the end of a table; a token whose id,
// position or type lies outside its table gets a row of NaN.
// Latency of three row gathers per wave and 8-byte-per-element traffic bound
// it: 6400 tokens of 768 columns take 12 us, where the position tensors of 64
// sequences alone cost 64 host synchronisations and launches.
//
// With `stats` one more block, the last, finds the longest, the shortest and the sum
// of the sequences' lengths, which the host wants before it can launch attention (as
// five launches ahead of this one, and an idle device until it knew, an encoder pass of
// 1 x 20 tokens took 909 us in place of 858, of 40 x 100 1721 for 1631).
constexpr int EMB_MAXV = 4;

// by one wave
__device__ __forceinline__ void length_stats(long* stats, const int* cu_seqlens,
                                             int num_seqs, int lane) {
  int longest = INT_MIN, shortest = INT_MAX;
  long sum = 0;
  for (int i = lane; i < num_seqs; i += 64) {
    const int len = (int)((unsigned int)cu_seqlens[i + 1] - (unsigned int)cu_seqlens[i]);
    longest = max(longest, len);
    shortest = min(shortest, len);
    sum += len;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    longest = max(longest, __shfl_xor(longest, off, 64));
    shortest = min(shortest, __shfl_xor(shortest, off, 64));
    sum += __shfl_xor(sum, off, 64);
  }
  if (lane == 0) {
    stats[0] = longest;
    stats[1] = shortest;
    stats[2] = sum;
  }
}

__global__ __launch_bounds__(256) void embed_layer_norm_kernel(
    short* __restrict__ out, const short* __restrict__ word,
    const short* __restrict__ pos_table, const short* __restrict__ type_table,
    const long* __restrict__ ids, const long* __restrict__ types,
    const int* __restrict__ cu_seqlens, const short* __restrict__ weight,
    const short* __restrict__ bias, const float eps, const int tokens,
    const int num_seqs, const int hidden, const int vocab, const int max_pos,
    const int num_types, long* __restrict__ stats) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (stats && blockIdx.x == gridDim.x - 1) {
    if (threadIdx.x < 64) length_stats(stats, cu_seqlens, num_seqs, lane);
    return;
  }
  if (t >= tokens) return;
  // last sequence that starts at or before the token
  const int first = cu_seqlens[0];
  int lo = 0, hi = num_seqs;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (cu_seqlens[mid] - first <= t) lo = mid;
    else hi = mid;
  }
  const int pos = t - (cu_seqlens[lo] - first);
  long id = ids[t], ty = types ? types[t] : 0;
  if (id < 0) id += vocab;
  if (ty < 0) ty += num_types;
  const bool ok = id >= 0 && id < vocab && pos >= 0 && pos < max_pos && ty >= 0 &&
                  ty < num_types;
  const int nvec = hidden >> 3;
  short8_t* ro = reinterpret_cast<short8_t*>(out) + (long)t * nvec;
  if (!ok) {
    short8_t bad;
#pragma unroll
    for (int j = 0; j < 8; ++j) bad[j] = 0x7fc0;  // NaN
    for (int i = lane; i < nvec; i += 64) ro[i] = bad;
    return;
  }
  const short8_t* rw = reinterpret_cast<const short8_t*>(word) + id * nvec;
  const short8_t* rp = reinterpret_cast<const short8_t*>(pos_table) + (long)pos * nvec;
  const short8_t* rt = reinterpret_cast<const short8_t*>(type_table) + ty * nvec;
  float x[EMB_MAXV][8];
  float sum = 0.f;
#pragma unroll
  for (int u = 0; u < EMB_MAXV; ++u) {
    const int i = lane + 64 * u;
    if (i < nvec) {
      const short8_t a = rw[i], b = rp[i], c = rt[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        x[u][j] = bf16_bits_to_float(a[j]) + bf16_bits_to_float(b[j]) +
                  bf16_bits_to_float(c[j]);
        sum += x[u][j];
      }
    }
  }
  const float mean = wave_reduce_sum(sum) / hidden;
  float sq = 0.f;
#pragma unroll
  for (int u = 0; u < EMB_MAXV; ++u)
    if (lane + 64 * u < nvec) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sq += (x[u][j] - mean) * (x[u][j] - mean);
    }
  const float rstd = rsqrtf(wave_reduce_sum(sq) / hidden + eps);
#pragma unroll
  for (int u = 0; u < EMB_MAXV; ++u) {
    const int i = lane + 64 * u;
    if (i < nvec) {
      const short8_t w = reinterpret_cast<const short8_t*>(weight)[i];
      const short8_t b = reinterpret_cast<const short8_t*>(bias)[i];
      short8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = float_to_bf16_bits((x[u][j] - mean) * rstd * bf16_bits_to_float(w[j]) +
                                  bf16_bits_to_float(b[j]));
      ro[i] = o;
    }
  }
}

}  // namespace

extern "C" {

hipError_t ks_embed_layer_norm(void* out, const void* word, const void* pos_table,
                               const void* type_table, const void* ids,
                               const void* types, const void* cu_seqlens,
                               const void* weight, const void* bias, float eps,
                               int tokens, int num_seqs, int hidden, int vocab,
                               int max_pos, int num_types, void* stats,
                               hipStream_t stream) {
  if (hidden % 8 != 0 || hidden > EMB_MAXV * 512 || num_seqs < 1)
    return hipErrorInvalidValue;
  const int blocks = (tokens + 3) / 4 + (stats ? 1 : 0);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(embed_layer_norm_kernel, dim3(blocks), dim3(256), 0, stream,
                     (short*)out, (const short*)word,
                     (const short*)pos_table, (const short*)type_table,
                     (const long*)ids, (const long*)types, (const int*)cu_seqlens,
                     (const short*)weight, (const short*)bias, eps, tokens,
                     num_seqs, hidden, vocab, max_pos, num_types, (long*)stats);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

hipError_t ks_layer_norm(void* out, const void* input, const void* weight,
                         const void* bias, float eps, int rows, int hidden,
                         hipStream_t stream) {
  return launch_layer_norm<false>(out, input, nullptr, weight, bias, eps, rows,
                                  hidden, stream);
}

hipError_t ks_fused_add_layer_norm(void* out, const void* input,
                                   const void* residual, const void* weight,
                                   const void* bias, float eps, int rows,
                                   int hidden, hipStream_t stream) {
  return launch_layer_norm<true>(out, input, residual, weight, bias, eps, rows,
                                 hidden, stream);
}

hipError_t ks_gelu(void* out, const void* input, long numel,
                   hipStream_t stream) {
  if (numel % 8 != 0) return hipErrorInvalidValue;
  long nvec = numel >> 3;
  if (nvec == 0) return hipSuccess;
  int grid = (int)((nvec + 255) / 256);
  if (grid > 2048) grid = 2048;
  hipLaunchKernelGGL(gelu_kernel, dim3(grid), dim3(256), 0, stream,
                     (short*)out, (const short*)input, nvec);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
}
