// Sampling kernels: greedy argmax and Gumbel-max temperature sampling.
//
// Gumbel-max: argmax(logit/T + G_i) with G_i = -log(-log(U_i)) samples the
// softmax(logit/T) distribution exactly, without materializing probabilities
// or sorting. Per-element U_i comes from a counter-based hash (seed, idx) so
// the kernel is stateless and hipGraph-replayable.
// (SURVEY.md §2.7 sampling row; north star: hand-written sampling kernel.)
#include "common.h"

namespace {

// xxhash-like 2x32 mix: deterministic per (seed, idx)
__device__ __forceinline__ unsigned int hash2(unsigned int a, unsigned int b) {
  unsigned int h = a * 0x9E3779B1u + b * 0x85EBCA77u + 0x165667B1u;
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  h ^= h >> 15;
  return h;
}

// One row of bf16 logits walked by a block of NT threads. The row starts at
// any 2-byte boundary (odd vocabularies): `head` elements up to the first
// 16-byte boundary, nvec vectors of 8, and a tail; head and tail (7 at most
// each) are one extra element of the first 16 threads.
template <int NT>
struct Bf16Row {
  const short* row;
  const short8_t* rv;
  int head, nvec, ex;  // ex: index of the extra element, -1 for none

  __device__ __forceinline__ Bf16Row(const short* p, int V) {
    row = p;
    const int tid = threadIdx.x;
    head = min(V, (int)(((16 - ((uintptr_t)p & 15)) & 15) >> 1));
    nvec = (V - head) >> 3;
    rv = reinterpret_cast<const short8_t*>(p + head);
    const int tail0 = head + nvec * 8;
    ex = tid < head ? tid : (tid >= 8 && tail0 + tid - 8 < V) ? tail0 + tid - 8 : -1;
  }
  // f(eight elements, index of the first) with four loads in flight, then
  // one(element, index) for this thread's extra element
  template <typename F, typename G>
  __device__ __forceinline__ void each8(F f, G one) const {
    int i = threadIdx.x;
    for (; i + 3 * NT < nvec; i += 4 * NT) {
      short8_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = rv[i + u * NT];
#pragma unroll
      for (int u = 0; u < 4; ++u) f(v[u], head + (i + u * NT) * 8);
    }
    for (; i < nvec; i += NT) f(rv[i], head + i * 8);
    if (ex >= 0) one(row[ex], ex);
  }
  template <typename F>
  __device__ __forceinline__ void each(F f) const {
    each8(
        [&](const short8_t& v, int i0) {
#pragma unroll
          for (int j = 0; j < 8; ++j) f(v[j], i0 + j);
        },
        f);
  }
};

// the block's largest value and its index (ties: the lower index) to out
template <int NT>
__device__ __forceinline__ void block_argmax(float best, int best_idx, long* out) {
  __shared__ float s_val[NT / 64];
  __shared__ int s_idx[NT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto merge = [&](float ov, int oi) {
    if (ov > best || (ov == best && oi < best_idx)) {
      best = ov;
      best_idx = oi;
    }
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    merge(__shfl_xor(best, off, 64), __shfl_xor(best_idx, off, 64));
  if (lane == 0) {
    s_val[wave] = best;
    s_idx[wave] = best_idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < NT / 64; ++w) merge(s_val[w], s_idx[w]);
    *out = best_idx;
  }
}

__device__ __forceinline__ float gumbel_noise(unsigned int seed, int idx) {
  const unsigned int h = hash2(seed, (unsigned int)idx);
  // u in (0,1): (h + 1) / 2^32
  const float u = ((float)h + 1.0f) * 2.3283064e-10f;
  return __logf(-__logf(u));
}

// logits bf16 [S, V]; one block of NT threads per row.
template <bool GUMBEL, int NT>
__global__ __launch_bounds__(NT) void argmax_kernel(
    long* __restrict__ out,            // [S]
    const short* __restrict__ logits,  // [S, V] bf16
    const float* __restrict__ temperatures,  // [S] (GUMBEL)
    const long* __restrict__ seeds,          // [S] (GUMBEL)
    const int V) {
  const int s = blockIdx.x;
  const short* row = logits + (long)s * V;
  const float inv_t = GUMBEL ? 1.f / fmaxf(temperatures[s], 1e-5f) : 1.f;
  const unsigned int seed = GUMBEL ? (unsigned int)(seeds[s] & 0xFFFFFFFF) : 0;

  float best = -1e38f;
  int best_idx = 0;
  // vectorized short8 loads over the vocab row
  const int nvec = V >> 3;
  const short8_t* rv = reinterpret_cast<const short8_t*>(row);
  for (int i = threadIdx.x; i < nvec; i += NT) {
    short8_t v = rv[i];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int idx = i * 8 + j;
      float val = bf16_bits_to_float(v[j]);
      if constexpr (GUMBEL) {
        val *= inv_t;
        val -= gumbel_noise(seed, idx);
      }
      if (val > best) {
        best = val;
        best_idx = idx;
      }
    }
  }
  // tail (V not divisible by 8)
  for (int idx = nvec * 8 + threadIdx.x; idx < V; idx += NT) {
    float val = bf16_bits_to_float(row[idx]);
    if constexpr (GUMBEL) {
      val *= inv_t;
      val -= gumbel_noise(seed, idx);
    }
    if (val > best) {
      best = val;
      best_idx = idx;
    }
  }
  block_argmax<NT>(best, best_idx, out + s);
}

// fp32 logits [S, V]: argmax of every bit, ties to the lower index; one block
// of 1024 threads per row. vec: rows start on 16-byte boundaries.
constexpr int AM_NT = 1024;

__global__ __launch_bounds__(AM_NT) void argmax_f32_kernel(
    long* __restrict__ out, const float* __restrict__ logits, const int V,
    const int vec) {
  const float* row = logits + (long)blockIdx.x * V;
  // finite: one of the modules this file is built into assumes finite math
  float best = -3.4e38f;
  int best_idx = 0;
  auto take = [&](float val, int idx) {
    // a thread's indexes only grow, so ">" keeps its lowest
    if (val > best) {
      best = val;
      best_idx = idx;
    }
  };
  int done = 0;
  if (vec) {
    const float4_t* rv = reinterpret_cast<const float4_t*>(row);
    const int nvec = V >> 2;
    int i = threadIdx.x;
    for (; i + 3 * AM_NT < nvec; i += 4 * AM_NT) {
      float4_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = rv[i + u * AM_NT];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < 4; ++c) take(v[u][c], (i + u * AM_NT) * 4 + c);
    }
    for (; i < nvec; i += AM_NT) {
      const float4_t v = rv[i];
#pragma unroll
      for (int c = 0; c < 4; ++c) take(v[c], i * 4 + c);
    }
    done = nvec * 4;
  }
  for (int i = done + threadIdx.x; i < V; i += AM_NT) take(row[i], i);
  __shared__ float s_val[AM_NT / 64];
  __shared__ int s_idx[AM_NT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  auto merge = [&](float ov, int oi) {
    if (ov > best || (ov == best && oi < best_idx)) {
      best = ov;
      best_idx = oi;
    }
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
    merge(__shfl_xor(best, off, 64), __shfl_xor(best_idx, off, 64));
  if (lane == 0) {
    s_val[wave] = best;
    s_idx[wave] = best_idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < AM_NT / 64; ++w) merge(s_val[w], s_idx[w]);
    out[blockIdx.x] = best_idx;
  }
}

// ---------------------------------------------------------------------------
// Fused top-k/top-p + Gumbel-max sampler, one block of 1024 threads per row.
//
// bf16 logits have 16-bit patterns that order monotonically once sign-flipped
// (key = bits<0 ? ~bits : bits|0x8000). The limits of top-k and top-p are
// found as keys from histograms, without a sort, and the last pass
// Gumbel-argmaxes over {key >= threshold}, which samples the truncated softmax
// exactly.
//
// All elements of one key have one probability, so counts per key are enough
// for the mass too: pass 2 counts the WIN keys below the row's largest (64 KB
// of LDS) and sums the whole row's mass in registers; a scan over the bins
// from the top then gives both limits exactly. WIN keys are 128 octaves below
// a positive maximum (all positive logits down to 2^-120 of it). Where a limit
// lies below the window (nearly flat rows, k of the order of the row) two
// coarser histograms find it: the keys' upper 12 bits, then the lower 4 inside
// the bin that the limit falls into.
//
// What bounds it: one pass of LDS atomics, an exponential per element and the
// three passes over the row, which come from the L2 and the memory-side cache.
// A histogram over the keys' upper byte puts a model's logits into half a
// dozen bins and serialises a wave's 64 adds, for count and mass each. Rows of
// N(0, 2.5) logits, top-k and top-p mixed, that form -> this one: 256 x 128256
// 704 -> 78 us, 256 x 32000 141 -> 34 us, 1 x 128256 465 -> 44 us; limits
// below the window (k of the order of the row) 702 -> 156 us. Holding the row
// in registers over the passes is not faster (80 us). Rows with nothing to cut
// go straight to the last pass (256 x 128256: 38 us; the plain kernel's 31 need
// the host to know that no row has a limit, a synchronisation of 15).
// ---------------------------------------------------------------------------
constexpr int RT = 1024;
constexpr int WIN = 16384;
constexpr int KBINS = 4096;

__device__ __forceinline__ unsigned int bf16_sort_key(short bits) {
  const unsigned short u = (unsigned short)bits;
  return (u & 0x8000u) ? (unsigned int)(unsigned short)~u
                       : (unsigned int)(u | 0x8000u);
}
__device__ __forceinline__ float key_value(unsigned int key) {
  return bf16_bits_to_float((short)((key & 0x8000u) ? (key & 0x7fffu) : ~key));
}

// Of bins 0, 1, ... with value(bin) each, PER per thread in order: the first
// bin at which the running sum reaches `target` goes to *bin and the sum
// before it to *above (neither is written if the total stays below). All
// threads of the block call it; the results can be read on return.
template <int PER, typename T, typename F>
__device__ __forceinline__ void find_bin(F value, T target, T* wave_sum, int* bin,
                                         T* above) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  T v[PER], own = 0;
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    v[j] = value(tid * PER + j);
    own += v[j];
  }
  T incl = own;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const T o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  T c = incl - own;
  for (int w = 0; w < wave; ++w) c += wave_sum[w];
  // a thread's end is the next one's start in exact sums only: in floating
  // point the first thread at or past the target is taken by the smaller bin
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    if (c < target && c + v[j] >= target) {
      if (atomicMin(bin, tid * PER + j) > tid * PER + j) *above = c;
    }
    c += v[j];
  }
  __syncthreads();
}

__global__ __launch_bounds__(RT) void topk_topp_sample_kernel(
    long* __restrict__ out,            // [S]
    const short* __restrict__ logits,  // [S, V] bf16
    const float* __restrict__ temperatures,
    const float* __restrict__ top_p,  // [S] (>=1 disables)
    const int* __restrict__ top_k,    // [S] (<=0 disables)
    const long* __restrict__ seeds,   // [S]
    const int V) {
  typedef unsigned long long u64;
  const int s = blockIdx.x;
  const float inv_t = 1.f / fmaxf(temperatures[s], 1e-5f);
  const float p = top_p[s];
  const int k = top_k[s];
  const unsigned int seed = (unsigned int)(seeds[s] & 0xFFFFFFFF);
  const bool use_k = (k > 0) && (k < V);
  bool use_p = p < 1.0f;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int NWV = RT / 64;
  constexpr int NONE = 0x7fffffff;

  __shared__ union {
    unsigned int win[WIN];
    struct {
      unsigned int cnt[KBINS];
      u64 mass[KBINS];
    } h;
  } lds;
  __shared__ unsigned int f_cnt[16];
  __shared__ u64 f_mass[16];
  __shared__ unsigned int s_key[NWV];
  __shared__ unsigned int s_bad[NWV];
  __shared__ double w_mass[NWV];
  __shared__ unsigned int w_cnt[NWV];
  __shared__ u64 w_fix[NWV];
  __shared__ int sh_bin[4];
  __shared__ unsigned int sh_above_k;
  __shared__ double sh_above_p;
  __shared__ u64 sh_above_f;

  const Bf16Row<RT> row(logits + (long)s * V, V);
  unsigned int thr = 0;
  if (use_k || use_p) {
    // ---- largest number (exp stability), and whether a mass can be formed ----
    unsigned int mk = 0;
    unsigned int bad = 0;  // a NaN or +inf: no mass, as its sum would be NaN
    row.each([&](short b, int) {
      const unsigned int mag = (unsigned short)b & 0x7fffu;
      if (mag > 0x7f80u || (unsigned short)b == 0x7f80u) bad = 1;
      else mk = max(mk, bf16_sort_key(b));
    });
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
      mk = max(mk, (unsigned int)__shfl_xor((int)mk, off, 64));
    bad = __ballot(bad != 0) != 0;
    if (lane == 0) {
      s_key[wave] = mk;
      s_bad[wave] = bad;
    }
    for (int i = tid; i < WIN; i += RT) lds.win[i] = 0;
    if (tid < 16) {
      f_cnt[tid] = 0;
      f_mass[tid] = 0;
    }
    if (tid < 4) sh_bin[tid] = NONE;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      mk = max(mk, s_key[w]);
      bad |= s_bad[w];
    }
    // all of them -inf: no mass either
    if (bad || mk <= 0x7fu) use_p = false;
    // with NaNs and infinities above it the largest number is not the
    // largest key, and the counts start at the top
    const unsigned int top = bad ? 0xffffu : mk;
    const float m = key_value(mk);
    auto weight = [&](float x) { return __expf((x - m) * inv_t); };

    // ---- counts per key in the window, mass of the row ----
    float z = 0.f;
    row.each([&](short b, int) {
      const unsigned int at = top - bf16_sort_key(b);
      if (at < WIN) atomicAdd(&lds.win[at], 1u);
      if (use_p) z += weight(bf16_bits_to_float(b));
    });
    double zz = z;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) zz += __shfl_xor(zz, off, 64);
    if (lane == 0) w_mass[wave] = zz;
    __syncthreads();
    zz = 0;
#pragma unroll
    for (int w = 0; w < NWV; ++w) zz += w_mass[w];
    __syncthreads();  // w_mass is written again below
    const double want_p = (double)p * zz;
    if (use_k)
      find_bin<WIN / RT, unsigned int>([&](int i) { return lds.win[i]; },
                                       (unsigned int)k, w_cnt, &sh_bin[0],
                                       &sh_above_k);
    if (use_p)
      find_bin<WIN / RT, double>(
          [&](int i) {
            const unsigned int n = lds.win[i];
            return n ? n * (double)weight(key_value(top - i)) : 0.0;
          },
          want_p, w_mass, &sh_bin[1], &sh_above_p);
    bool far_k = use_k, far_p = use_p && want_p > 0;
    if (use_k && sh_bin[0] != NONE) {
      thr = top - sh_bin[0];
      far_k = false;
    }
    if (far_p && sh_bin[1] != NONE) {
      thr = max(thr, top - sh_bin[1]);
      far_p = false;
    }
    // the larger threshold wins, so a limit below the window matters only if
    // the other one is not inside it
    if ((far_k || far_p) && thr == 0) {
      constexpr float ONE = 1099511627776.0f;  // mass in 2^-40 of the largest term
      auto fixed = [&](short b) {
        return (u64)(fminf(weight(bf16_bits_to_float(b)), 1.f) * ONE + 0.5f);
      };
      __syncthreads();
      for (int i = tid; i < KBINS; i += RT) {
        lds.h.cnt[i] = 0;
        lds.h.mass[i] = 0;
      }
      if (tid < 4) sh_bin[tid] = NONE;
      __syncthreads();
      u64 zf = 0;
      row.each([&](short b, int) {
        const int hi = KBINS - 1 - (bf16_sort_key(b) >> 4);
        if (far_k) atomicAdd(&lds.h.cnt[hi], 1u);
        if (far_p) {
          const u64 f = fixed(b);
          zf += f;
          atomicAdd(&lds.h.mass[hi], f);
        }
      });
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) zf += __shfl_xor(zf, off, 64);
      if (lane == 0) w_fix[wave] = zf;
      __syncthreads();
      zf = 0;
#pragma unroll
      for (int w = 0; w < NWV; ++w) zf += w_fix[w];
      __syncthreads();
      const u64 want_f = max((u64)1, (u64)((double)p * (double)zf));
      if (far_k)
        find_bin<KBINS / RT, unsigned int>([&](int i) { return lds.h.cnt[i]; },
                                           (unsigned int)k, w_cnt, &sh_bin[0],
                                           &sh_above_k);
      if (far_p)
        find_bin<KBINS / RT, u64>([&](int i) { return lds.h.mass[i]; }, want_f,
                                  w_fix, &sh_bin[1], &sh_above_f);
      const int bk = sh_bin[0], bp = sh_bin[1];
      // lower bits inside the two boundary bins
      row.each([&](short b, int) {
        const unsigned int key = bf16_sort_key(b);
        const int hi = KBINS - 1 - (key >> 4);
        if (hi == bk) atomicAdd(&f_cnt[15 - (key & 15)], 1u);
        if (hi == bp) atomicAdd(&f_mass[15 - (key & 15)], fixed(b));
      });
      __syncthreads();
      if (bk != NONE) {
        const unsigned int want = (unsigned int)k - sh_above_k;
        find_bin<1, unsigned int>([&](int i) { return i < 16 ? f_cnt[i] : 0u; }, want,
                                  w_cnt, &sh_bin[2], &sh_above_k);
        thr = ((KBINS - 1 - bk) << 4) | (15 - sh_bin[2]);
      }
      if (bp != NONE) {
        const u64 want = want_f - sh_above_f;
        find_bin<1, u64>([&](int i) { return i < 16 ? f_mass[i] : (u64)0; }, want,
                         w_fix, &sh_bin[3], &sh_above_f);
        thr = max(thr, (unsigned int)((KBINS - 1 - bp) << 4) | (15 - sh_bin[3]));
      }
    }
  }

  // ---- Gumbel-argmax over the surviving set: the lanes of a wave go through
  // their own survivors, so a sparse set costs few rounds of hash and logs ----
  float best = -1e38f;
  int best_idx = 0;
  auto take = [&](short b, int i) {
    // top-k of one is the greedy choice, ties included: no noise
    float val = bf16_bits_to_float(b) * inv_t;
    if (k != 1) val -= gumbel_noise(seed, i);
    if (val > best || (val == best && i < best_idx)) {
      best = val;
      best_idx = i;
    }
  };
  row.each8(
      [&](const short8_t& v, int i0) {
        if (thr == 0) {  // nothing cut: every element, without the detour
#pragma unroll
          for (int j = 0; j < 8; ++j) take(v[j], i0 + j);
          return;
        }
        unsigned int in = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) in |= (bf16_sort_key(v[j]) >= thr ? 1u : 0u) << j;
        while (in) {
          const int j = __builtin_ctz(in);
          in &= in - 1;
          short b = v[0];
#pragma unroll
          for (int q = 1; q < 8; ++q) b = j == q ? v[q] : b;
          take(b, i0 + j);
        }
      },
      [&](short b, int i) {
        if (bf16_sort_key(b) >= thr) take(b, i);
      });
  block_argmax<RT>(best, best_idx, out + s);
}

// 1024 threads for rows past 64k elements (256 rows of 128256, greedy 24.7 ->
// 12.3 us, with noise 36.5 -> 30.8); shorter rows are over before a block that
// size has merged its waves (256 x 32000, greedy: 5.9 us with 256 threads, 7.0
// with 1024)
template <bool GUMBEL>
void launch_argmax(void* out, const void* logits, const void* temperatures,
                   const void* seeds, int num_seqs, int vocab, hipStream_t stream) {
  if (vocab > 65536)
    hipLaunchKernelGGL((argmax_kernel<GUMBEL, 1024>), dim3(num_seqs), dim3(1024), 0,
                       stream, (long*)out, (const short*)logits,
                       (const float*)temperatures, (const long*)seeds, vocab);
  else
    hipLaunchKernelGGL((argmax_kernel<GUMBEL, 256>), dim3(num_seqs), dim3(256), 0,
                       stream, (long*)out, (const short*)logits,
                       (const float*)temperatures, (const long*)seeds, vocab);
}

}  // namespace

extern "C" {

hipError_t ks_greedy_sample(void* out, const void* logits, int num_seqs,
                            int vocab, int is_f32, hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  if (is_f32) {
    const int vec = vocab % 4 == 0 && ((uintptr_t)logits % 16) == 0;
    hipLaunchKernelGGL(argmax_f32_kernel, dim3(num_seqs), dim3(AM_NT), 0, stream,
                       (long*)out, (const float*)logits, vocab, vec);
    HIP_CHECK_KERNEL();
    return hipSuccess;
  }
  launch_argmax<false>(out, logits, nullptr, nullptr, num_seqs, vocab, stream);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

hipError_t ks_gumbel_sample(void* out, const void* logits,
                            const void* temperatures, const void* top_k,
                            const void* seeds, int num_seqs, int vocab,
                            hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  // sampling from the whole row: top_k is not read
  launch_argmax<true>(out, logits, temperatures, seeds, num_seqs, vocab, stream);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

hipError_t ks_topk_topp_sample(void* out, const void* logits,
                               const void* temperatures, const void* top_p,
                               const void* top_k, const void* seeds,
                               int num_seqs, int vocab, hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  hipLaunchKernelGGL(topk_topp_sample_kernel, dim3(num_seqs), dim3(RT), 0,
                     stream, (long*)out, (const short*)logits,
                     (const float*)temperatures, (const float*)top_p,
                     (const int*)top_k, (const long*)seeds, vocab);
  HIP_CHECK_KERNEL();
  return hipSuccess;
}
}
