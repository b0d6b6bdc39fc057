// Sampling kernels: greedy argmax and Gumbel-max temperature sampling.
//
// Gumbel-max: argmax(logit/T + G_i) with G_i = -log(-log(U_i)) samples the
// softmax(logit/T) distribution exactly, without materializing probabilities
// or sorting. Per-element U_i comes from a counter-based hash (seed, idx) so
// the kernel is stateless and hipGraph-replayable.
#include "common.h"
#include "decode_step.h"

#include <type_traits>

namespace {

// xxhash-like 2x32 mix, deterministic per (seed, idx): hash_end of
// hash_start(seed) + idx * HASH_STEP
constexpr unsigned int HASH_STEP = 0x85EBCA77u;

__device__ __forceinline__ unsigned int hash_start(unsigned int seed) {
  return seed * 0x9E3779B1u + 0x165667B1u;
}
// all but the last step, which leaves the upper 15 bits as they are
constexpr unsigned int HASH_LOW = 0x1ffffu;
__device__ __forceinline__ unsigned int hash_upper(unsigned int h) {
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  return h;
}
__device__ __forceinline__ unsigned int hash_end(unsigned int h) {
  h = hash_upper(h);
  return h ^ (h >> 15);
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
  // group(vectors, integral_constant of their number (4 or 1), index of the
  // first element; the vectors are NT * 8 elements apart) by whole waves, with
  // four loads in flight; rest(vector, index of its first element) for the last
  // nvec % 64; then one(element, index) for this thread's extra element
  template <typename F, typename R, typename G>
  __device__ __forceinline__ void groups(F group, R rest, G one) const {
    const int whole = nvec & ~63;
    int i = threadIdx.x;
    for (; i + 3 * NT < whole; i += 4 * NT) {
      short8_t v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = rv[i + u * NT];
      group(v, std::integral_constant<int, 4>{}, head + i * 8);
    }
    for (; i < whole; i += NT) {
      const short8_t v[1] = {rv[i]};
      group(v, std::integral_constant<int, 1>{}, head + i * 8);
    }
    if (i < nvec) rest(rv[i], head + i * 8);
    if (ex >= 0) one(row[ex], ex);
  }
  // f(eight elements, index of the first)
  template <typename F, typename G>
  __device__ __forceinline__ void each8(F f, G one) const {
    groups(
        [&](const short8_t* v, auto count, int i0) {
#pragma unroll
          for (int u = 0; u < decltype(count)::value; ++u) f(v[u], i0 + u * NT * 8);
        },
        f, one);
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

// the block's largest value and its index (ties: the lower index), to all threads or
// the first
template <int NT, bool ALL>
__device__ __forceinline__ void block_best(float& best, int& best_idx) {
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
  if (ALL || threadIdx.x == 0) {
    for (int w = ALL ? 0 : 1; w < NT / 64; ++w) merge(s_val[w], s_idx[w]);
  }
}
template <int NT>
__device__ __forceinline__ void block_argmax(float best, int best_idx, long* out) {
  block_best<NT, false>(best, best_idx);
  if (threadIdx.x == 0) *out = best_idx;
}

__device__ __forceinline__ float noise_of_hash(unsigned int h) {
  // u in (0,1): (h + 1) / 2^32, which rounds to 1 for the last 128 hashes: their
  // noise would be infinite, and win the row whatever the logit
  const float u = fminf(((float)h + 1.0f) * 2.3283064e-10f, 0.99999994f);
  return __logf(-__logf(u));
}
// Whether x / T + G can reach the best score that the wave has seen. With u = 1 -
// r / 2^32 the noise is at most ln(2^32 / r), so an element whose r is above 2^32
// exp(x / T - best) cannot. r's float pattern is a logarithm of it to within 0.09,
// so the test is a multiply-add, two conversions and a compare beside the hash, in
// place of two logarithms.
//
// Margin in log2: over all 2^32 hashes with r past 4096 (below, an element always
// passes) pattern, u's rounding and the two hardware logarithms are off by 0.031 at
// most; the rest of the 0.15 and the term in |best| are for the fp32 sums of scores.
struct GumbelBound {
  static constexpr float ONE = 8388608.f;  // 2^23: 1 in log2 as a pattern
  float c1, c0 = __builtin_bit_cast(float, 0x7f800000);  // every number passes at first

  __device__ __forceinline__ explicit GumbelBound(float inv_t)
      : c1(inv_t * 1.44269504f * ONE) {
    asm("" : "+v"(c0));  // (infinite, which fast math would take for impossible)
  }
  __device__ __forceinline__ bool passes(float x, unsigned int hash) const {
    const float r = (float)(~hash);
    // At least the pattern of 4096, and within the range of an int. The product of a
    // low x is past the range of a float, as c0 is after such a best: in one rounding
    // the sum is infinite for every number and NaN, which is taken for the lower
    // limit, for an x of -inf.
    const float t = __builtin_amdgcn_fmed3f(__builtin_fmaf(x, c1, c0), 1166016512.f, 2.1e9f);
    return __builtin_bit_cast(int, r) <= (int)t;
  }
  // by a whole wave
  __device__ __forceinline__ void raise(float best) {
    const float b = fminf(wave_reduce_max(best), 1e30f);
    c0 = (32.f + 127.f - b * 1.44269504f + (0.15f + 2e-6f * fabsf(b))) * ONE;
  }
};

// A thread's part of argmax(x / T + G) over a whole row, ties to the lower index.
// Bound by arithmetic, 20 operations an element with the hash's two multiplies at
// a quarter of the rate. 256 x 128256: 37.7 us with two logarithms for every
// element, 26.9 with the bound; 256 x 32000 17.1 -> 13.1. Blocks of few waves walk
// short rows, where the score to beat is found too late to pay for the bound.
template <int NT>
__device__ __forceinline__ void gumbel_row(const Bf16Row<NT>& row, const float inv_t,
                                           const unsigned int seed, float& best,
                                           int& best_idx) {
  const unsigned int h0 = hash_start(seed);
  GumbelBound bound(inv_t);
  bool started = false;
  auto take = [&](float x, unsigned int h, int i) {
    const float val = x * inv_t - noise_of_hash(h);
    if (val > best || (val == best && i < best_idx)) {
      best = val;
      best_idx = i;
    }
  };
  auto vec = [&](const short8_t& v, const int i0) {
    const unsigned int hi = h0 + (unsigned int)i0 * HASH_STEP;
    if (!started) {  // the wave's first elements give it a score to beat
      take(bf16_bits_to_float(v[0]), hash_end(hi), i0);
      bound.raise(best);
      started = true;
    }
    unsigned int in = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      in |= (bound.passes(bf16_bits_to_float(v[j]), hash_end(hi + j * HASH_STEP)) ? 1u : 0u)
            << j;
    if (__ballot(in != 0)) {
      while (in) {
        const int j = __builtin_ctz(in);
        in &= in - 1;
        short b = v[0];
#pragma unroll
        for (int q = 1; q < 8; ++q) b = j == q ? v[q] : b;
        take(bf16_bits_to_float(b), hash_end(hi + j * HASH_STEP), i0 + j);
      }
      bound.raise(best);
    }
  };
  // the wave's maximum takes whole waves: the rest is evaluated in full
  row.groups(
      [&](const short8_t* v, auto count, int i0) {
#pragma unroll
        for (int u = 0; u < decltype(count)::value; ++u) vec(v[u], i0 + u * NT * 8);
      },
      [&](const short8_t& v, int i0) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          take(bf16_bits_to_float(v[j]),
               hash_end(h0 + (unsigned int)(i0 + j) * HASH_STEP), i0 + j);
      },
      [&](short b, int i) {
        take(bf16_bits_to_float(b), hash_end(h0 + (unsigned int)i * HASH_STEP), i);
      });
}

// A greedy row's share of the next step's inputs: their addresses do not wait for the
// token, so they are fetched ahead of the row. A launch of their own took 4 us
// by itself and 1 of a captured step (1 row 446.5 -> 445.3, 24 rows 532.2 -> 531.0).
struct RowNext {
  long pos = 0;
  int slot = 0;
  __device__ __forceinline__ RowNext(const NextStep& to, long row) {
    if (!to.ids) return;
    pos = to.positions[row] + 1;
    slot = next_slot(to, row, pos);
  }
};

// logits bf16 [S, V]; one block of NT threads per row.
template <bool GUMBEL, int NT>
__global__ __launch_bounds__(NT) void argmax_kernel(
    long* __restrict__ out,            // [S]
    const short* __restrict__ logits,  // [S, V] bf16
    const float* __restrict__ temperatures,  // [S] (GUMBEL)
    const long* __restrict__ seeds,          // [S] (GUMBEL)
    const int V, const NextStep next) {
  const int s = blockIdx.x;
  const short* row = logits + (long)s * V;
  const RowNext own(next, s);

  const float inv_t = GUMBEL ? 1.f / fmaxf(temperatures[s], 1e-5f) : 1.f;
  const unsigned int seed = GUMBEL ? (unsigned int)(seeds[s] & 0xFFFFFFFF) : 0;

  float best = -1e38f;
  int best_idx = 0;
  if constexpr (GUMBEL && NT >= 1024) {
    gumbel_row<NT>(Bf16Row<NT>(row, V), inv_t, seed, best, best_idx);
  } else {
    auto take = [&](short b, int idx) {
      float val = bf16_bits_to_float(b);
      if constexpr (GUMBEL) {
        val *= inv_t;
        val -= noise_of_hash(hash_end(hash_start(seed) + (unsigned int)idx * HASH_STEP));
      }
      if (val > best) {  // a thread's indexes only grow
        best = val;
        best_idx = idx;
      }
    };
    // vectorized short8 loads over the vocab row
    const int nvec = V >> 3;
    const short8_t* rv = reinterpret_cast<const short8_t*>(row);
    for (int i = threadIdx.x; i < nvec; i += NT) {
      const short8_t v = rv[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) take(v[j], i * 8 + j);
    }
    // tail (V not divisible by 8)
    for (int idx = nvec * 8 + threadIdx.x; idx < V; idx += NT) take(row[idx], idx);
  }
  block_best<NT, false>(best, best_idx);
  if (threadIdx.x == 0) {
    out[s] = best_idx;
    if (next.ids) write_next(next, s, best_idx, own.pos, own.slot);
  }
}

// fp32 logits [S, V]: argmax of every bit, ties to the lower index; one block
// of 1024 threads per row. vec: rows start on 16-byte boundaries.
constexpr int AM_NT = 1024;

__global__ __launch_bounds__(AM_NT) void argmax_f32_kernel(
    long* __restrict__ out, const float* __restrict__ logits, const int V,
    const int vec, const NextStep next) {
  const float* row = logits + (long)blockIdx.x * V;
  const RowNext own(next, blockIdx.x);
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
    if (next.ids) write_next(next, blockIdx.x, best_idx, own.pos, own.slot);
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
// The usual row takes one pass for all of it ("first pass"): counts of the keys
// between 2^-16 and 2^16 of either sign in 8193 bins (those closer to 0 share one)
// and the first and last bin, by 16-bit packed operations while the row comes from
// memory. The mass is formed from the counts, and the bins are scanned from the
// row's largest, 1024 at a time, until the higher limit is found; one scan nearly
// always does. Where fewer than k elements have a bin, the others being masked, all
// of those survive. Where a limit, or mass that counts, lies at 0, a pass more tells
// the zeros apart. Rows with NaNs or numbers above 2^16, and those where numbers
// between 0 and 2^-16 of either sign decide, go through the passes above.
//
// The last pass queues a wave's survivors in LDS and evaluates them 64 at a time,
// so a set of any density costs what it holds. Of a large one it forms every hash and
// queues the few whose noise can exceed what some of them nearly surely reach.
//
// What bounds it: the first pass runs at memory speed (8 operations an element
// hide under it), the last at the vector units' and the queue's. Rows of N(0, 2.5)
// logits, one per compute unit (us, three passes / this): 256 x 128256 top-p 0.9 75
// / 37, top-k 50 49 / 29, both 52 / 30; 15 x 128256 66 / 31, 40 / 20, 45 / 22; 256 x
// 32000 33 / 20, 23 / 14, 29 / 16; limits below zero 131 / 68 (a histogram by the
// keys' upper byte took 704 at 256 x 128256). 256 x 128256, top-k 50 of 20 numbers, the
// rest masked, 306 / 38; half of the row 0, top-p 0.99 212 / 111 (all of it 0: 137 /
// 162, the counts of one bin one after the other). Holding the row in registers over the
// passes was no faster.
// ---------------------------------------------------------------------------
constexpr int RT = 1024;
constexpr int WIN = 16384;
constexpr int KBINS = 4096;

// First pass: a 16-bit pattern as a signed number in the logits' order, with the
// patterns of +-2^-16 .. 0 taken out of the middle: bin FSPAN - that, FBINS in all
constexpr int FSPAN = 4096, FBINS = 2 * FSPAN + 1;
constexpr short NEAR_HI = 0x377f, NEAR_LO = -0x3780;
constexpr int MINUS_INF_BIN = FSPAN + 0x7f81 + NEAR_LO;
typedef short short2_v __attribute__((ext_vector_type(2)));
typedef unsigned short ushort2_v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ short2_v ordered(short2_v b) {
  const short2_v sign = b >> 15;
  return b ^ __builtin_bit_cast(short2_v, __builtin_bit_cast(ushort2_v, sign) >> 1);
}
__device__ __forceinline__ ushort2_v first_bin(short2_v s) {
  const short2_v lo = {NEAR_LO, NEAR_LO}, hi = {NEAR_HI, NEAR_HI};
  const short2_v mid = __builtin_elementwise_min(__builtin_elementwise_max(s, lo), hi);
  return __builtin_bit_cast(ushort2_v, (short2_v)(short2_v{FSPAN, FSPAN} - (s - mid)));
}
// the number of an ordered pattern, and the ordered pattern of a bin
__device__ __forceinline__ float ordered_value(int s) {
  return bf16_bits_to_float((short)(s ^ ((s >> 15) & 0x7fff)));
}
__device__ __forceinline__ int bin_ordered(int bin) {
  const int d = FSPAN - bin;
  return d > 0 ? d + NEAR_HI : d < 0 ? d + NEAR_LO : 0;
}

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

// Elements whose scores can reach the cut (in log2), queued by a whole wave as its
// vectors pass by. With 1 - u = r / 2^32 the noise is at most ln(2^32 / r), so an
// element whose r is above 2^32 exp(x / T - cut) cannot. The upper 15 bits of r decide,
// against the largest x of a lane's eight, and r below 2^17 always passes: beside the
// hash that is half an operation an element, where GumbelBound takes eight.
// Margin: u's rounding and the two hardware logarithms are off by 0.031 in log2 at most
// from r 4096 on; the rest, and the term in the cut, are for the fp32 scores.
struct CandidateQueue {
  uint2* queue;
  int most;  // entries
  float c2, c0;
  unsigned int h0;
  int queued = 0;

  __device__ __forceinline__ CandidateQueue(uint2* q, int n, float c2_, float cut, unsigned int h)
      : queue(q), most(n), c2(c2_), c0(32.25f + 4e-6f * fabsf(cut) - cut), h0(h) {}
  __device__ __forceinline__ bool full() const { return queued > most; }
  __device__ __forceinline__ void add8(const short8_t& v, int i0) {
    short2_v m = {-32768, -32768};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      m = __builtin_elementwise_max(m, ordered(short2_v{v[2 * q], v[2 * q + 1]}));
    const float x = ordered_value(max(m.x, m.y));
    const float t = __builtin_amdgcn_fmed3f(
        __builtin_amdgcn_exp2f(__builtin_fmaf(x, c2, c0)), 131072.f, 4294967040.f);
    const unsigned int least = ~((unsigned int)t | HASH_LOW);
    const unsigned int hi = h0 + (unsigned int)i0 * HASH_STEP;
    unsigned int h[8], last = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      h[j] = hash_upper(hi + j * HASH_STEP);
      last = max(last, h[j]);
    }
    if (!__ballot(last >= least)) return;
    unsigned int in = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) in |= (h[j] >= least ? 1u : 0u) << j;
    for (;;) {  // one of each lane's at a time
      const unsigned long long set = __ballot(in != 0);
      if (!set) break;
      const int j = __builtin_ctz(in | 0x100);
      short b = v[0];
#pragma unroll
      for (int q = 1; q < 8; ++q) b = j == q ? v[q] : b;
      const int at = __builtin_amdgcn_mbcnt_hi(
          (unsigned int)(set >> 32), __builtin_amdgcn_mbcnt_lo((unsigned int)set, queued));
      if (in && at < most)
        queue[at] = uint2{(unsigned int)(i0 + j), (unsigned int)(unsigned short)b << 16};
      queued += __builtin_popcountll(set);
      in &= in - 1;
    }
  }
};

__global__ __launch_bounds__(RT) void topk_topp_sample_kernel(
    long* __restrict__ out,            // [S]
    const short* __restrict__ logits,  // [S, V] bf16
    const float* __restrict__ temperatures,
    const float* __restrict__ top_p,  // [S] (>=1 and <=0 disable)
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
  bool use_p = p > 0.f && p < 1.f;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  constexpr int NWV = RT / 64;
  constexpr int NONE = 0x7fffffff;
  constexpr int QUEUE = 63 + 8 * 64;  // survivors of a wave on their way

  __shared__ union {
    unsigned int win[WIN];
    struct {
      unsigned int cnt[KBINS];
      u64 mass[KBINS];
    } h;
    uint2 queue[NWV][QUEUE];
  } lds;
  __shared__ unsigned int f_cnt[16];
  __shared__ u64 f_mass[16];
  __shared__ unsigned int s_key[NWV];
  __shared__ unsigned int s_bad[NWV];
  __shared__ double w_mass[NWV];
  __shared__ unsigned int w_cnt[NWV];
  __shared__ u64 w_fix[NWV];
  __shared__ int sh_bin[4];
  __shared__ unsigned int sh_above_k, sh_live;
  __shared__ double sh_above_p;
  __shared__ u64 sh_above_f;

  const Bf16Row<RT> row(logits + (long)s * V, V);
  unsigned int thr = 0;
  // where many survive: how many, and log2 of a score that some of them exceed
  unsigned int live = 0;
  bool by_mass = false;
  float cut = 0.f;
  if (use_k || use_p) {
    // ---- first pass: counts per bin, extremes, mass ----
    for (int i = tid; i < FBINS; i += RT) lds.win[i] = 0;
    if (tid < 4) sh_bin[tid] = NONE;
    if (tid == 0) sh_live = 0;
    __syncthreads();
    const float c2 = inv_t * 1.44269504f;
    ushort2_v lo2 = {65535, 65535}, hi2 = {0, 0};  // first and last bin
    auto add = [&](short2_v b) {
      const ushort2_v at = first_bin(ordered(b));
      lo2 = __builtin_elementwise_min(lo2, at);
      hi2 = __builtin_elementwise_max(hi2, at);
      if (at.x < FBINS) atomicAdd(&lds.win[at.x], 1u);
      if (at.y < FBINS) atomicAdd(&lds.win[at.y], 1u);
    };
    auto add8 = [&](const short8_t& v, int) {
#pragma unroll
      for (int q = 0; q < 4; ++q) add(short2_v{v[2 * q], v[2 * q + 1]});
    };
    row.each8(add8, [&](short b, int) {
      const unsigned short at = first_bin(ordered(short2_v{b, b})).x;
      lo2 = __builtin_elementwise_min(lo2, ushort2_v{at, at});
      hi2 = __builtin_elementwise_max(hi2, ushort2_v{at, at});
      if (at < FBINS) atomicAdd(&lds.win[at], 1u);
    });
    unsigned int lo = min((unsigned int)lo2.x, (unsigned int)lo2.y);
    unsigned int hi = max((unsigned int)hi2.x, (unsigned int)hi2.y);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, (unsigned int)__shfl_xor((int)lo, off, 64));
      hi = max(hi, (unsigned int)__shfl_xor((int)hi, off, 64));
    }
    if (lane == 0) {
      s_key[wave] = lo;
      s_bad[wave] = hi;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      lo = min(lo, s_key[w]);
      hi = max(hi, s_bad[w]);
    }
    // past the last bin come numbers below -2^16, -inf, NaNs, then what is above
    // 2^16; the largest number has a bin
    const bool direct = hi <= MINUS_INF_BIN && lo < FBINS;
    const float most = direct ? ordered_value(bin_ordered(lo)) : 0.f;
    auto weight_of_bin = [&](int bin) {
      return (double)__builtin_amdgcn_exp2f((ordered_value(bin_ordered(bin)) - most) * c2);
    };
    if (direct) {
      double zz = 0;
      if (use_p) {
#pragma unroll
        for (int i = 0; i < (FBINS + RT - 1) / RT; ++i) {
          const int bin = tid + i * RT;
          const unsigned int n = bin < FBINS ? lds.win[bin] : 0u;
          if (n) zz += n * weight_of_bin(bin);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) zz += __shfl_xor(zz, off, 64);
        if (lane == 0) w_mass[wave] = zz;
        __syncthreads();
        zz = 0;
#pragma unroll
        for (int w = 0; w < NWV; ++w) zz += w_mass[w];
      }
      const double want = (double)p * zz;
      unsigned int over_k = 0;  // elements and mass of the bins before
      double over_p = 0;
      for (int b0 = lo; b0 < FBINS; b0 += RT) {
        __syncthreads();  // the sums of the round before are read
        const int bin = b0 + tid;
        const unsigned int n = bin < FBINS ? lds.win[bin] : 0u;
        const double m = use_p && n ? n * weight_of_bin(bin) : 0.0;
        unsigned int nk = n;
        double mp = m;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const unsigned int a = __shfl_up(nk, off, 64);
          const double b = __shfl_up(mp, off, 64);
          if (lane >= off) {
            nk += a;
            mp += b;
          }
        }
        if (lane == 63) {
          w_cnt[wave] = nk;
          w_mass[wave] = mp;
        }
        __syncthreads();
        unsigned int ck = over_k + nk - n;
        double cp = over_p + (mp - m);
#pragma unroll
        for (int w = 0; w < NWV; ++w) {
          ck += w < wave ? w_cnt[w] : 0u;
          cp += w < wave ? w_mass[w] : 0.0;
          over_k += w_cnt[w];
          over_p += w_mass[w];
        }
        // the first bin at which the running sum reaches its target; in
        // floating point a thread's end need not be the next one's start
        if (use_k && n && ck < (unsigned int)k && ck + n >= (unsigned int)k) {
          atomicMin(&sh_bin[0], bin);
          if (bin == FSPAN) sh_above_k = ck;
        }
        if (use_p && n && cp < want && cp + m >= want) {
          atomicMin(&sh_bin[1], bin);
          if (bin == FSPAN) sh_above_p = cp;
        }
        __syncthreads();
        // the smaller bin is the higher limit, and what is not found yet lies below
        const int found = min(sh_bin[0], sh_bin[1]);
        if (found != NONE) {
          if (bin == found) sh_live = ck + n;
          break;
        }
      }
      const int bin = min(sh_bin[0], sh_bin[1]);
      // Numbers below -2^16 and -inf have no bin. Where the largest stands 40 / ln 2
      // scaled logits above them, no noise (-3.1 to 16.7) brings one up, and their mass
      // has to be nothing beside the row's.
      const double below = V * (double)__builtin_amdgcn_exp2f((-65536.f - most) * c2);
      const bool whole =
          hi < FBINS || ((most + 65536.f) * c2 >= 40.f && below <= 3e-8);
      // Numbers closer to 0 than 2^-16 share a bin. With a limit in it, or their mass
      // (known to 2^-16 / T of it) not to be left uncertain, zeros are told apart.
      const unsigned int near = lds.win[FSPAN];
      const double weight0 = near ? weight_of_bin(FSPAN) : 0.0;
      auto known = [&](unsigned int n) {
        return !use_p || n * weight0 * c2 * 1.6e-5 <= 3e-8 * zz;
      };
      bool sure = known(near);
      // positive numbers down to the last before 0, to the last +0, to the last -0
      unsigned int to[3] = {0, 0, 0};
      if (near && (bin == FSPAN || !sure)) {
        row.each([&](short b, int) {
          const unsigned int u = (unsigned short)b;
          to[0] += u - 1 < (unsigned int)NEAR_HI ? 1u : 0u;
          to[1] += u == 0u ? 1u : 0u;
          to[2] += u == 0x8000u ? 1u : 0u;
        });
        unsigned int* const sums[3] = {w_cnt, s_key, s_bad};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
#pragma unroll
          for (int off = 32; off > 0; off >>= 1)
            to[i] += (unsigned int)__shfl_xor((int)to[i], off, 64);
          if (lane == 0) sums[i][wave] = to[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          to[i] = i ? to[i - 1] : 0u;
#pragma unroll
          for (int w = 0; w < NWV; ++w) to[i] += sums[i][w];
        }
        sure = known(near - (to[2] - to[0]));
      }
      // (a limit of top-k above all that has no bin needs no mass)
      if (sure && (whole || (bin != NONE && !use_p))) {
        if (bin == FSPAN) {
          const double k_left = sh_bin[0] == FSPAN ? (double)k - sh_above_k : 1e30;
          const double p_left = sh_bin[1] == FSPAN ? want - sh_above_p : 1e30;
          auto reached = [&](unsigned int n) { return k_left <= n || p_left <= n * weight0; };
          if (!reached(to[0])) thr = reached(to[1]) ? 0x8000u : reached(to[2]) ? 0x7fffu : 0u;
        } else {  // no limit among the bins: all that is in them
          thr = (unsigned int)(bin_ordered(bin == NONE ? FBINS - 1 : bin) + 32768);
          // with the mass known, elements above its logarithm less 2.5 are Poisson with
          // a mean of 12
          if (use_p && bin == sh_bin[1]) {
            by_mass = true;
            cut = most * c2 + __builtin_amdgcn_logf((float)want) - 2.5f * 1.44269504f;
          }
        }
      }
    }
    __syncthreads();
    if (by_mass) live = sh_live;  // (written after the scan's last barrier)
  }
  if ((use_k || use_p) && thr == 0) {
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

  // ---- Gumbel-argmax over the surviving set ----
  float best = -1e38f;
  int best_idx = 0;
  if (thr == 0 && k != 1) {
    gumbel_row<RT>(row, inv_t, seed, best, best_idx);
  } else {
    const unsigned int h0 = hash_start(seed);
    GumbelBound bound(inv_t);
    // top-k of one is the greedy choice, ties included: no noise
    auto take = [&](float x, unsigned int h, int i) {
      const float val = k == 1 ? x * inv_t : x * inv_t - noise_of_hash(h);
      if (val > best || (val == best && i < best_idx)) {
        best = val;
        best_idx = i;
      }
    };
    auto take_one = [&](short b, int i) {
      if (bf16_sort_key(b) >= thr)
        take(bf16_bits_to_float(b), hash_end(h0 + (unsigned int)i * HASH_STEP), i);
    };
    __syncthreads();  // the counts are read
    // Where many survive, each element's hash is formed and the few that can exceed the
    // cut are evaluated; where few do, queueing the survivors costs less (us, queue /
    // this, 256 rows: 128256 logits, a fifth surviving 41.5 / 37.0, a third 44.1 / 36.9,
    // 7 % 37.6 / 37.8; 32000 logits 20.6 / 20.0, 21.6 / 19.9, 18.9 / 20.4; 16 x 128256
    // 35.7 / 31.3, 38.3 / 31.2).
    if (live > (unsigned int)V / 10) {
      CandidateQueue could(lds.queue[wave], QUEUE, inv_t * 1.44269504f, cut, h0);
      row.groups(
          [&](const short8_t* v, auto count, int i0) {
            if (could.full()) return;
#pragma unroll
            for (int u = 0; u < decltype(count)::value; ++u)
              could.add8(v[u], i0 + u * RT * 8);
          },
          [&](const short8_t& v, int i0) {
#pragma unroll
            for (int j = 0; j < 8; ++j) take_one(v[j], i0 + j);
          },
          take_one);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      for (int at = lane; at < min(could.queued, QUEUE); at += 64) {
        const uint2 e = lds.queue[wave][at];
        take_one((short)(e.y >> 16), (int)e.x);
      }
      float most = could.full() ? 3e38f : best;
      int most_idx = best_idx;
      block_best<RT, true>(most, most_idx);
      // (not so if a queue ran over or, by chance, nothing exceeds the cut)
      if (most < 1e38f && most * 1.44269504f >= cut) {
        if (tid == 0) out[s] = most_idx;
        return;
      }
      __syncthreads();  // block_best is called again
    }
    uint2* queue = lds.queue[wave];
    int queued = 0;
    auto drain = [&](int from) {  // 64 of the queue, by a whole wave
      const uint2 e = queue[from + lane];
      const float x = __builtin_bit_cast(float, e.y);
      const unsigned int h = hash_end(h0 + e.x * HASH_STEP);
      if (__ballot(k == 1 || bound.passes(x, h))) {
        take(x, h, (int)e.x);
        if (k != 1) bound.raise(best);
      }
    };
    // key >= thr as one unsigned comparison per half of a dword: the patterns
    // of positive limits are ordered once the sign is flipped, those of negative
    // ones once all bits are (positive numbers come out on top either way)
    const bool pos = thr & 0x8000u;
    const unsigned int flip = pos ? 0x80008000u : 0xffffffffu;
    const unsigned int lim = thr;
    row.groups(
        [&](const short8_t* v, auto count, int i0) {
#pragma unroll
          for (int u = 0; u < decltype(count)::value; ++u) {
            const uint4 d = __builtin_bit_cast(uint4, v[u]);
            const unsigned int dw[4] = {d.x, d.y, d.z, d.w};
            ushort2_v m = {0, 0};
#pragma unroll
            for (int q = 0; q < 4; ++q)
              m = __builtin_elementwise_max(
                  m, __builtin_bit_cast(ushort2_v, dw[q] ^ flip));
            if (!__ballot(max((unsigned int)m.x, (unsigned int)m.y) >= lim)) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
              const unsigned int w = dw[j / 2] ^ flip;
              const bool in = j & 1 ? w >= lim << 16
                                    : (unsigned short)w >= (unsigned short)lim;
              const u64 set = __ballot(in);
              if (set) {
                if (in)
                  queue[queued + __builtin_amdgcn_mbcnt_hi(
                                     (unsigned int)(set >> 32),
                                     __builtin_amdgcn_mbcnt_lo((unsigned int)set, 0))] =
                      uint2{(unsigned int)(i0 + u * RT * 8 + j),
                            j & 1 ? dw[j / 2] & 0xffff0000u : dw[j / 2] << 16};
                queued += __builtin_popcountll(set);
              }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            while (queued >= 64) drain(queued -= 64);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          }
        },
        [&](const short8_t& v, int i0) {
#pragma unroll
          for (int j = 0; j < 8; ++j) take_one(v[j], i0 + j);
        },
        take_one);
    if (lane < queued) {
      const uint2 e = queue[lane];
      take(__builtin_bit_cast(float, e.y), hash_end(h0 + e.x * HASH_STEP), (int)e.x);
    }
  }
  block_argmax<RT>(best, best_idx, out + s);
}

// 256 threads, or 1024: a row's time is the latency of its loads one after the
// other, which more threads shorten, but a block of 1024 merges its waves for longer
// and two fit a compute unit. Rows of more than 65536 take 1024 (256 x 128256, greedy
// 24.7 -> 12.7 us, with noise 36.5 -> 25.8). Shorter ones with noise stay with 256, which
// evaluate every element (256 x 32000 10.5 us, 11.9 with 512 and the bound). Greedy ones
// take 1024 as long as the rows come to one or two a unit (us with 256 / 1024: 1, 256
// rows of 18000 4.2 / 4.1, 4.7 / 4.8, of 32000 5.4 / 4.6, 6.1 / 5.3; 300, 512 rows of 28000
// 5.8 / 6.2, 7.8 / 6.8, of 32000 8.6 / 6.9, 9.0 / 7.5; 1024 rows of 32000 12.2 / 14.1; 256 rows
// of 14000 4.3 / 4.6).
bool wide_argmax(bool noise, int num_seqs, int vocab) {
  if (vocab > 65536) return true;
  return !noise && num_seqs <= 512 && vocab > (num_seqs <= 256 ? 18000 : 30000);
}

template <bool GUMBEL>
void launch_argmax(void* out, const void* logits, const void* temperatures,
                   const void* seeds, int num_seqs, int vocab, const NextStep& next,
                   hipStream_t stream) {
  if (wide_argmax(GUMBEL, num_seqs, vocab))
    hipLaunchKernelGGL((argmax_kernel<GUMBEL, 1024>), dim3(num_seqs), dim3(1024), 0,
                       stream, (long*)out, (const short*)logits,
                       (const float*)temperatures, (const long*)seeds, vocab, next);
  else
    hipLaunchKernelGGL((argmax_kernel<GUMBEL, 256>), dim3(num_seqs), dim3(256), 0,
                       stream, (long*)out, (const short*)logits,
                       (const float*)temperatures, (const long*)seeds, vocab, next);
}

}  // namespace

extern "C" {

static hipError_t greedy_rows(void* out, const void* logits, int num_seqs, int vocab,
                              int is_f32, const NextStep& next, hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  if (is_f32) {
    const int vec = vocab % 4 == 0 && ((uintptr_t)logits % 16) == 0;
    hipLaunchKernelGGL(argmax_f32_kernel, dim3(num_seqs), dim3(AM_NT), 0, stream,
                       (long*)out, (const float*)logits, vocab, vec, next);
  } else {
    launch_argmax<false>(out, logits, nullptr, nullptr, num_seqs, vocab, next, stream);
  }
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

hipError_t ks_greedy_sample(void* out, const void* logits, int num_seqs,
                            int vocab, int is_f32, hipStream_t stream) {
  return greedy_rows(out, logits, num_seqs, vocab, is_f32, NextStep{}, stream);
}

// the greedy tokens, and the next decode step's inputs from them
hipError_t ks_greedy_advance(void* out, const void* logits, int num_seqs, int vocab,
                             int is_f32, void* ids, void* positions, void* context_lens,
                             void* slots, const void* tables, long table_stride, int width,
                             int block, hipStream_t stream) {
  if (width < 1 || block < 1 || !ids) return hipErrorInvalidValue;
  const NextStep next{(long*)ids,  (long*)positions,   (int*)context_lens,
                      (int*)slots, (const int*)tables, table_stride, width, block};
  return greedy_rows(out, logits, num_seqs, vocab, is_f32, next, stream);
}

hipError_t ks_gumbel_sample(void* out, const void* logits,
                            const void* temperatures, const void* top_k,
                            const void* seeds, int num_seqs, int vocab,
                            hipStream_t stream) {
  if (num_seqs == 0) return hipSuccess;
  // sampling from the whole row: top_k is not read
  launch_argmax<true>(out, logits, temperatures, seeds, num_seqs, vocab, NextStep{}, stream);
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
