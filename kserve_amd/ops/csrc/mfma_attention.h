// Paged and flat softmax attention on the bf16 matrix cores: the kernels behind
// attention_prefill.hip and attention_decode.hip (bf16 queries) and the bf16
// pages of attention_f32.hip (fp32 queries and softmax weights).
//
// PARTS is how many bf16 parts an fp32 operand enters with: three hold its 24
// bits exactly (high, middle, low: 8 bits each), so the products with bf16 keys
// and values are exact and everything is summed in fp32.
#pragma once

#include "common.h"
#include "mfma_layouts.h"

namespace {
namespace mfma_attn {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.44269504088896340736f;
constexpr float MASKED = -3e38f;
constexpr float NO_MAX = -1e30f;  // above MASKED: an all-masked tile adds 0
constexpr int PAGE = 16;

// where K and V rows come from
enum Src {
  ROWS_DMA,   // flat rows, 16-byte aligned: loaded straight into LDS
  ROWS_REG,   // flat rows at any alignment: through registers
  PAGES_DMA,  // bf16 pages of 16 tokens, 16-byte aligned: straight into LDS
  PAGES_REG,  // bf16 pages at any alignment: through registers
  PAGES_FP8,  // E4M3 pages, widened to bf16 on the way
};

// 16-byte chunk that chunk c of row r of a tile sits at. K fragments: 16
// consecutive rows at one chunk must hit different banks; V fragments: 4
// consecutive rows of 32 bytes each (a pair of chunks stays a pair).
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  return D == 128 ? (r & 15) : ((r >> 1) & 7);
}
template <int D>
__device__ __forceinline__ int v_swz(int r) {
  return D == 128 ? (r & 7) << 1 : ((r >> 1) & 3) << 1;
}

__device__ __forceinline__ f32x16_t mfma32(bf16x8_t a, bf16x8_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// What the launchers hand the kernels as their scale: scores are masked before
// they are scaled, and the scaled mask has to give weight 0. Below 1e-30 all
// scores are level whatever the scale.
inline float score_scale(float scale) {
  return fabsf(scale) < 1e-30f ? copysignf(1e-30f, scale) : scale;
}

// x as the sum of three bf16 numbers, exactly
struct Split3 {
  __bf16 hi, mid, lo;
  __device__ __forceinline__ explicit Split3(float x) {
    hi = (__bf16)x;
    const float r1 = x - (float)hi;
    mid = (__bf16)r1;
    lo = (__bf16)(r1 - (float)mid);
  }
};

// two numbers as bf16
struct Rounded2 {
  unsigned int bits;
  __device__ __forceinline__ Rounded2(float x, float y) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    bits = __builtin_bit_cast(unsigned int, __builtin_convertvector((float2_t{x, y}), bf16x2_t));
  }
  __device__ __forceinline__ float first() const { return __uint_as_float(bits << 16); }
  __device__ __forceinline__ float second() const { return __uint_as_float(bits & 0xffff0000u); }
};

// what the fp32 form adds to plain attention
struct Extra {
  const short* gate;  // [T, H] bf16 (row stride gate_stride): output * sigmoid
  long gate_stride;
  const float* sink;  // [H]: one more term exp(sink) in the denominator
  int chunk;          // a query sees its own block of that many positions
  int out_f32;        // fp32 output (else bf16)
};

// first position that a query at `pos` sees
__device__ __forceinline__ int low_of(int pos, int window, int chunk) {
  return chunk > 0 ? pos / chunk * chunk : window > 0 ? max(pos - window + 1, 0) : 0;
}

__device__ __forceinline__ float sigmoid_gate(const Extra& x, long tok, int head) {
  return x.gate ? 1.f / (1.f + expf(-bf16_bits_to_float(x.gate[tok * x.gate_stride + head])))
                : 1.f;
}

__device__ __forceinline__ void store4(void* out, long at, f32x4_t v, int f32) {
  if (f32) {
    *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(out) + at) = v;
  } else {
    short4_t w;
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = float_to_bf16_bits(v[r]);
    *reinterpret_cast<short4_t*>(reinterpret_cast<short*>(out) + at) = w;
  }
}

// larger of a lane's value and its partner's in the other half of the wave
__device__ __forceinline__ float half_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(
      __float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// eight E4M3 bytes as bf16 (exact)
__device__ __forceinline__ short8_t widen_fp8(uint2 x) {
  short8_t o;
  const unsigned int w[2] = {x.x, x.y};
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const float2_t lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[d], false);
    const float2_t hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)w[d], true);
    o[d * 4 + 0] = float_to_bf16_bits(lo[0]);
    o[d * 4 + 1] = float_to_bf16_bits(lo[1]);
    o[d * 4 + 2] = float_to_bf16_bits(hi[0]);
    o[d * 4 + 3] = float_to_bf16_bits(hi[1]);
  }
  return o;
}

constexpr int KT = 64;      // keys per tile
constexpr int NWAVES = 4;
constexpr int QW = 32;      // queries per wave

struct PrefillArgs {
  void* out;          // [T, Hq, D]
  const void* q;      // [T, Hq, D] bf16 (PARTS 1) or fp32, row stride sq
  const void* k;      // [T, Hkv, D] rows (stride sk) or pages [NB, Hkv, 16, D]
  const void* v;      // likewise, page rows sv apart
  const int* cu_q;          // [S+1]
  const int* ctx_lens;      // [S] keys of a sequence (pages)
  const int* block_tables;  // [S, max_nb] (pages, row stride max_nb)
  int Hq, Hkv, max_nb;
  int hpb;  // query heads per block: 1, 2 or 4, divides the group
  float scale;
  long sq, sk, sv;
  int window;
  Extra x;
  // keys in n_splits parts (pages, one part per value): sums of the parts
  int n_splits;
  long rows;        // T * Hq
  float* part_out;  // [n_splits, T, Hq, D]
  float* part_ml;   // [n_splits, T, Hq, 2]: exponent, sum of weights or NO_KEYS
};
constexpr float NO_KEYS = -1.f;  // of a part without a tile, which writes no sums

// While a wave has products to issue it goes ahead of the other on its SIMD: that one's
// exponentials fill the cycles between, where by age a wave among its vector
// instructions keeps the products waiting (us: 1 x 8191 tokens 542 -> 533, 2 x 1000 queries
// over 13000 keys 366 -> 348, fp32 scores 4 x 2000 204 -> 198; only around the second
// product 550 and 362, the second above the first 541 and 357, the other way about 557 and
// 360, the vector part ahead 576 and 367). Not heads of 64, whose units have four waves a
// SIMD (64 texts of 123 tokens 19.0 / 19.2).
template <int D, int FIRST>
__device__ __forceinline__ void go_first() {
  if constexpr (D == 128) __builtin_amdgcn_s_setprio(FIRST);
}

template <int D, int SRC, bool CAUSAL, bool WIN, int PARTS = 1>
__global__ __launch_bounds__(256, 2) void prefill_attention_kernel(
    const PrefillArgs p) {
  // key blocks of 32 that go through softmax together: with three parts the
  // operands of one fill the registers
  constexpr int NKB = PARTS == 1 ? 2 : 1;
  constexpr bool PAGED = SRC >= PAGES_DMA;
  constexpr bool DMA = SRC == ROWS_DMA || SRC == PAGES_DMA;
  constexpr int CPR = D / 8;          // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;       // rows per wave-wide 16-byte load
  constexpr int NI = 16 / RPI;        // such loads per wave and tile (K or V)
  constexpr int TILE = KT * D;
  constexpr int KC = D / 16;          // contraction chunks of Q K^T
  constexpr int DB = D / 32;          // 32-column blocks of the output

  constexpr bool SPLITS = PAGED && PARTS == 1;
  const int seq = SPLITS ? blockIdx.z / p.n_splits : blockIdx.z;
  const int split = SPLITS ? blockIdx.z % p.n_splits : 0;
  const int q_start = p.cu_q[seq];
  const int q_len = p.cu_q[seq + 1] - q_start;
  const int qpb = NWAVES * QW / p.hpb;  // queries per block
  // the last tiles have the most keys: they start first
  const int tile_base = (gridDim.y - 1 - blockIdx.y) * qpb;
  if (tile_base >= q_len) return;
  const int len = PAGED ? p.ctx_lens[seq] : q_len;  // keys
  const int start_pos = len - q_len;                // position of query 0
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int head = blockIdx.x * p.hpb + wave % p.hpb;
  const int kvh = blockIdx.x * p.hpb / (p.Hq / p.Hkv);
  const int q0 = tile_base + wave / p.hpb * QW;  // the wave's first query
  const int half = lane >> 5;

  __shared__ __attribute__((aligned(16))) short lds[2][2][TILE];  // [buffer][K, V]

  // The scale's sign goes into the query, exactly. With three parts it is applied to
  // the scores: as a branch between products and softmax it keeps the compiler from
  // moving one into the other, for which there are no registers.
  float c2 = p.scale * LOG2E;
  const bool flip = c2 < 0.f;
  c2 = fabsf(c2);

  // ---- queries: B operands, 8 consecutive columns per lane ----
  bf16x8_t qf[PARTS][KC];
  {
    const int qrow = min(q0 + (lane & 31), q_len - 1);
    const long at = (long)(q_start + qrow) * p.sq + (long)head * D + half * 8;
    if constexpr (PARTS == 1) {
      const short* qp = reinterpret_cast<const short*>(p.q) + at;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        short8_t x = *reinterpret_cast<const short8_t*>(qp + c * 16);
        if (flip) x ^= (short)0x8000;
        qf[0][c] = __builtin_bit_cast(bf16x8_t, x);
      }
    } else {
      const float* qp = reinterpret_cast<const float*>(p.q) + at;
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          const f32x4_t x = *reinterpret_cast<const f32x4_t*>(qp + c * 16 + j);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const Split3 w(x[e]);
            qf[0][c][j + e] = w.hi;
            qf[1][c][j + e] = w.mid;
            qf[2][c][j + e] = w.lo;
          }
        }
    }
  }

  // ---- key range ----
  const int last_q = min(tile_base + qpb, q_len) - 1;
  const int hi = CAUSAL ? min(len, start_pos + last_q + 1) : len;
  auto low = [&](int pos) { return low_of(pos, p.window, p.x.chunk); };
  const int lo = WIN ? max(0, low(start_pos + tile_base)) : 0;
  int t_lo = lo / KT;
  int t_hi = (hi + KT - 1) / KT;
  if (SPLITS && p.n_splits > 1) {
    const int per = (t_hi - t_lo + p.n_splits - 1) / p.n_splits;
    t_lo += split * per;
    t_hi = min(t_hi, t_lo + per);
  }
  const int pos_lo = start_pos + q0;
  const int pos_hi = start_pos + min(q0 + QW, q_len) - 1;
  const int my_pos = start_pos + q0 + (lane & 31);
  // first visible key of the wave's first and last query and of this lane's
  const int low_lo = WIN ? low(pos_lo) : 0, low_hi = WIN ? low(pos_hi) : 0;
  const int my_low = WIN ? low(my_pos) : 0;

  // ---- staging: wave w brings rows 16 w .. 16 w + 15 of a tile (one page);
  // rows past the keys repeat the last one (their weights are 0, their values
  // finite) ----
  const int* bt = PAGED ? p.block_tables + (long)seq * p.max_nb : nullptr;
  const int lrow = lane / CPR, lchunk = lane % CPR;
  auto group_of = [&](int t) { return min(t * KT + wave * 16, len - 1); };
  auto page_of = [&](int t) { return PAGED ? bt[group_of(t) >> 4] : 0; };
  // A scalar base per tile and 32-bit lane offsets (the launchers see to strides
  // below 2^26): tiles with all their keys cost no vector arithmetic, where 64-bit
  // addresses per lane and load took 500 of a tile's 1800 vector cycles. (As buffer
  // loads they would leave the compiler's waits for a wave's LDS reads one after the
  // other: 1 x 8191 tokens 564 -> 550 us, 64 texts of 123 tokens with heads of 64 13.3 ->
  // 14.1; the check of the waits ahead of the barriers reads the global form.)
  constexpr int ES = SRC == PAGES_FP8 ? 1 : 2;
  const int krs = PAGED && PARTS == 1 ? D : (int)p.sk;  // bf16 queries: whole rows
  const int vrs = PAGED && PARTS == 1 ? D : (int)p.sv;
  // (three parts leave no registers for them: there they are formed per tile)
  constexpr bool KEEP = PARTS == 1;
  unsigned int koff[NI], voff[NI];
#pragma unroll
  for (int i = 0; KEEP && i < NI; ++i) {
    const int r = i * RPI + lrow;
    koff[i] = (unsigned int)(r * krs + (lchunk ^ k_swz<D>(r)) * 8) * ES;
    voff[i] = (unsigned int)(r * vrs + (lchunk ^ v_swz<D>(r)) * 8) * ES;
  }
  auto base_of = [&](const void* base, int stride, int g0, int page) {
    const long at = PAGED ? ((long)page * p.Hkv + kvh) * PAGE * stride
                          : (long)(q_start + g0) * stride + kvh * D;
    return reinterpret_cast<const char*>(base) + at * ES;
  };
  uint2 raw8[SRC == PAGES_FP8 ? 2 * NI : 1];
  short8_t raw16[!DMA && SRC != PAGES_FP8 ? 2 * NI : 1];
  // DMA: fills buffer `buf`; otherwise the rows wait in registers for commit()
  auto stage_rows = [&](const char* kb, const char* vb, auto k_at, auto v_at, int buf) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const unsigned int ka = k_at(i), va = v_at(i);
      if constexpr (DMA) {
        const int at = (wave * 16 + i * RPI) * D;
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned int*>(kb + ka),
                                         reinterpret_cast<unsigned int*>(&lds[buf][0][at]),
                                         16, 0, 0);
        __builtin_amdgcn_global_load_lds(reinterpret_cast<const unsigned int*>(vb + va),
                                         reinterpret_cast<unsigned int*>(&lds[buf][1][at]),
                                         16, 0, 0);
      } else if constexpr (SRC == PAGES_FP8) {
        raw8[2 * i] = *reinterpret_cast<const uint2*>(kb + ka);
        raw8[2 * i + 1] = *reinterpret_cast<const uint2*>(vb + va);
      } else {
        raw16[2 * i] = *reinterpret_cast<const short8_t*>(kb + ka);
        raw16[2 * i + 1] = *reinterpret_cast<const short8_t*>(vb + va);
      }
    }
  };
  auto stage = [&](int t, int page, int buf) {
    const int g0 = PAGED ? group_of(t) & ~15 : group_of(t);
    const char* kb = base_of(p.k, krs, g0, page);
    const char* vb = base_of(p.v, vrs, g0, page);
    if (KEEP && (t + 1) * KT <= len)
      stage_rows(kb, vb, [&](int i) { return koff[i]; }, [&](int i) { return voff[i]; }, buf);
    else
      stage_rows(
          kb, vb,
          [&](int i) {
            const int r = i * RPI + lrow;
            return (unsigned int)(min(r, len - 1 - g0) * krs + (lchunk ^ k_swz<D>(r)) * 8) * ES;
          },
          [&](int i) {
            const int r = i * RPI + lrow;
            return (unsigned int)(min(r, len - 1 - g0) * vrs + (lchunk ^ v_swz<D>(r)) * 8) * ES;
          },
          buf);
  };
  auto commit = [&](int buf) {
    if constexpr (!DMA) {
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int at = (wave * 16 + i * RPI) * D + lane * 8;
#pragma unroll
        for (int kv = 0; kv < 2; ++kv) {
          short8_t x;
          if constexpr (SRC == PAGES_FP8) x = widen_fp8(raw8[2 * i + kv]);
          else x = raw16[2 * i + kv];
          *reinterpret_cast<short8_t*>(&lds[buf][kv][at]) = x;
        }
      }
    }
  };

  // ---- operand addresses inside a tile (elements) ----
  const int krow = lane & 31;
  int kaddr[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c)
    kaddr[c] = krow * D + ((2 * c + half) ^ k_swz<D>(krow)) * 8;
  // transposing load: lane i of 16 brings key i/4, columns 4 (i%4) .. + 3 of a
  // 4 x 16 block and receives column i of its four keys
  const int ti = lane & 15;
  const int vrow = half * 4 + (ti >> 2);
  int vaddr[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    vaddr[b] = vrow * D +
               (((4 * b + ((lane >> 4) & 1) * 2 + ((ti & 3) >> 1)) ^ v_swz<D>(vrow)) * 8) +
               (ti & 1) * 4;

  // Weights are 2^(score c2 - mc). mc follows the row's largest score only once it
  // is passed by 2^8: the sums have the room, and the rescaling of the output that
  // each new maximum of any of the 32 rows costs becomes rare.
  constexpr float ROOM = 8.f;
  float mc = fmaxf(NO_MAX * c2, -3e38f), l = 0.f;
  f32x16_t o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[b][r] = 0.f;

  if (t_lo < t_hi) stage(t_lo, page_of(t_lo), 0);
  int page = t_lo + 1 < t_hi ? page_of(t_lo + 1) : 0;
  commit(0);

  for (int t = t_lo; t < t_hi; ++t) {
    const int buf = (t - t_lo) & 1;
    // The barrier publishes tile t, and does not wait for this wave's LDS-direct
    // loads of it. The wait that the compiler puts ahead of the LDS reads is on
    // the path of a wave that computes; one without queries here has none.
    if constexpr (DMA) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t + 1 < t_hi) {
      stage(t + 1, page, buf ^ 1);
      if (PAGED && t + 2 < t_hi) page = page_of(t + 2);
    }
    const int t0 = t * KT;
    const bool mine = q0 < q_len && (!CAUSAL || t0 <= pos_hi) &&
                      (!WIN || t0 + KT - 1 >= low_lo);
    if (mine) {
      const short* kt = lds[buf][0];
      const short* vt = lds[buf][1];
#pragma unroll
      for (int kg = 0; kg < 2; kg += NKB) {
      f32x16_t s[NKB];
      if constexpr (PARTS == 1) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
        // both key blocks' chains side by side, keys read ahead of the products
        go_first<D, 1>();
#pragma unroll
        for (int c = 0; c < KC; ++c)
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
            s[kb] = mfma32(*reinterpret_cast<const bf16x8_t*>(kt + kb * 32 * D + kaddr[c]),
                           qf[0][c], s[kb]);
        constexpr int READS = NKB * KC, AHEAD = READS < 6 ? READS : 6;
        __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);  // LDS reads
#pragma unroll
        for (int i = 0; i < READS - AHEAD; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // matrix products
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
        go_first<D, 0>();
      } else {
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        f32x16_t rest;  // the products with the query's lower parts
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = rest[r] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(
              kt + (kg + kb) * 32 * D + kaddr[c]);
          rest = mfma32(a, qf[PARTS - 1][c], rest);
          rest = mfma32(a, qf[PARTS - 2][c], rest);
          s[kb] = mfma32(a, qf[0][c], s[kb]);
        }
        s[kb] += rest;
      }
      if (flip) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb) s[kb] = -s[kb];
      }
      }
      // register r of block kb: key 32 kb + (r & 3) + 8 (r / 4) + 4 half
      if (t0 + KT > len || (CAUSAL && t0 + KT - 1 > pos_lo) ||
          (WIN && t0 < low_hi)) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = t0 + 32 * (kg + kb) + (r & 3) + 8 * (r >> 2) + 4 * half;
            const bool ok = key < len && (!CAUSAL || key <= my_pos) &&
                            (!WIN || key >= my_low);
            s[kb][r] = ok ? s[kb][r] : MASKED;
          }
      }
      float mx = s[0][0];
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
      mx = half_max(mx) * c2;
      if (__any(mx > mc + ROOM)) {
        const float mn = fmaxf(mc, mx);
        const float f = __builtin_amdgcn_exp2f(mc - mn);
        mc = mn;
        l *= f;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[b][r] *= f;
      }
      bf16x8_t pf[PARTS][NKB * 2];
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float w = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], c2, -mc));
          sum += w;
          if constexpr (PARTS == 1) {
            pf[0][kb * 2 + (r >> 3)][r & 7] = (__bf16)w;
          } else {
            const Split3 w3(w);
            pf[0][kb * 2 + (r >> 3)][r & 7] = w3.hi;
            pf[1][kb * 2 + (r >> 3)][r & 7] = w3.mid;
            pf[2][kb * 2 + (r >> 3)][r & 7] = w3.lo;
          }
        }
      l += sum;
      go_first<D, 1>();
#pragma unroll
      for (int kc = 0; kc < NKB * 2; ++kc)
#pragma unroll
        for (int b = 0; b < DB; ++b) {
          typedef __attribute__((address_space(3))) s16x4_t lds4_t;
          const short* a0 = vt + (kg * 2 + kc) * 16 * D + vaddr[b];
          const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)a0);
          const s16x4_t v1 =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)(a0 + 8 * D));
          union {
            s16x4_t h[2];
            bf16x8_t v;
          } a;
          a.h[0] = v0;
          a.h[1] = v1;
#pragma unroll
          for (int part = PARTS - 1; part >= 0; --part)
            o[b] = mfma32(a.v, pf[part][kc], o[b]);
        }
      go_first<D, 0>();
      }
    }
    if (t + 1 < t_hi) commit(buf ^ 1);
  }

  if (q0 >= q_len) return;
  const int qrow = q0 + (lane & 31);
  l = half_sum(l);
  if (qrow >= q_len) return;
  const long tok = q_start + qrow;
  if (SPLITS && p.n_splits > 1) {
    const long row = split * p.rows + tok * p.Hq + head;
    const bool none = t_lo >= t_hi;
    if (half == 0)
      *reinterpret_cast<float2_t*>(p.part_ml + row * 2) = float2_t{mc, none ? NO_KEYS : l};
    if (none) return;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = o[b][g * 4 + r];
        store4(p.part_out, row * D + half * 4 + b * 32 + g * 8, w, 1);
      }
    return;
  }
  float inv;
  if constexpr (PARTS == 1) {
    inv = l > 0.f ? 1.f / l : 0.f;
  } else {
    if (p.x.sink) {
      // exp(sink) joins the denominator; the larger of the two maxima scales
      const float sl = p.x.sink[head] * LOG2E, ml = mc, top = fmaxf(ml, sl);
      const float f = exp2f(ml - top);
      l = l * f + exp2f(sl - top);
      inv = f / l;
    } else {
      inv = 1.f / l;
    }
    inv *= sigmoid_gate(p.x, tok, head);
  }
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4_t w;
#pragma unroll
      for (int r = 0; r < 4; ++r) w[r] = o[b][g * 4 + r] * inv;
      store4(p.out, (tok * p.Hq + head) * D + half * 4 + b * 32 + g * 8, w,
             PARTS == 1 ? 0 : p.x.out_f32);
    }
}

// Key parts of a prefill over pages. A block walks its tiles of 64 keys one after
// the other, 1.4 us each where a compute unit has one block and 2.2 with two, so
// few queries behind a long context leave most of the chip waiting; parts cost a
// launch and fp32 sums that are written and read. The estimate of both is taken
// from what was measured (32 / 8 heads, us, one part / chosen): 4 x 48 queries
// after 12900 keys 294 / 70, 3 x 56 after 1844 42 / 25, 2 x 200 after 14000 321 / 119,
// 700 after 5000 121 / 86, 32 after 600 17.5 / 13.8; 4 x 382 after 462 stays one).
inline int prefill_splits(long blocks, int tiles, long rows) {
  if (blocks <= 0 || tiles <= 0 || rows <= 0) return 1;
  int best = 1;
  double least = 0;
  for (int n = 1; n <= 32 && n <= tiles; ++n) {
    const long all = blocks * n, rounds = (all + 511) / 512;
    const double tile = all <= 256 ? 1.4 : 2.2 * rounds;
    const double us = (tiles + n - 1) / n * tile + 2.0 * rounds +
                      (n > 1 ? 4.0 + rows * 128 * 4.0 * 2 * n / 3e6 : 0.0);
    if (n == 1 || us < 0.95 * least) {
      best = n;
      least = us;
    }
  }
  return best;
}

// over the four lanes that share a column (lane & 15)
__device__ __forceinline__ float column_max(float x) {
  const unsigned int u = __float_as_uint(x);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned int v = __float_as_uint(
      fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float column_sum(float x) {
  x += __shfl_xor(x, 16, 64);
  return x + __shfl_xor(x, 32, 64);
}

// the pages of a sequence that are read, in pairs, and how they are split
struct Range {
  int first, last;  // page numbers
  int pairs;
  int splits;       // of the launched ones, those with work
  int per;          // pairs per split
};
__device__ __forceinline__ Range page_range(int ctx, int window, int chunk,
                                            int n_splits, int waves) {
  Range r;
  const int lo = ctx > 0 ? low_of(ctx - 1, window, chunk) : 0;
  r.first = lo / PAGE;
  r.last = (ctx - 1) / PAGE;
  r.pairs = ctx > 0 ? (r.last - r.first) / 2 + 1 : 0;
  // a pair per wave at least
  r.splits = max(1, min(n_splits, (r.pairs + waves - 1) / waves));
  r.per = (r.pairs + r.splits - 1) / r.splits;
  return r;
}

__device__ __forceinline__ uint4 load16_nt(const char* from) {
  typedef unsigned int u4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(
      uint4, __builtin_nontemporal_load(reinterpret_cast<const u4*>(from)));
}

// Waves of a block that share a context, and page pairs of a split from which on the
// launches with four use all of them: bf16 pages a pair for each (the LDS of the other
// two is taken in any case).
constexpr int WAVES = 2;
constexpr int deep_pairs(int src) { return src == PAGES_FP8 ? 16 : 2 * WAVES; }

struct DecodeArgs {
  void* out;                // [S, H, D]
  const void* q;            // [S, H, D] bf16 (PARTS 1) or fp32, row stride sq
  const void* k_cache;      // [NB, Hkv, 16, D], rows sk elements apart
  const void* v_cache;      // likewise, sv
  const int* block_tables;  // [S, max_blocks]
  const int* ctx_lens;      // [S]
  float scale;
  int H, Hkv, group, max_blocks;
  long sq;
  int n_splits;
  float* part_out;  // [S, H, n_splits, D]
  float* part_ml;   // [S, H, n_splits, 2]
  int window;
  long sk, sv;
  const int* cu_q;  // [S+1] first token of a sequence (null: sequence s's is s)
  Extra x;
};

// query token of sequence s, -1 if it has none in this batch
__device__ __forceinline__ int token_of(const DecodeArgs& p, int s) {
  if (!p.cu_q) return s;
  return p.cu_q[s + 1] > p.cu_q[s] ? p.cu_q[s] : -1;
}

// what a (token, head)'s weighted values are multiplied by: their largest
// exponent m (log2) and the sum of the weights relative to it
template <int PARTS>
__device__ __forceinline__ float final_factor(const DecodeArgs& p, long tok, int head,
                                              float m, float sum) {
  if constexpr (PARTS == 1) {
    return sum > 0.f ? 1.f / sum : 0.f;
  } else {
    float f = 1.f;
    if (p.x.sink) {
      const float sl = p.x.sink[head] * LOG2E, top = fmaxf(m, sl);
      f = exp2f(m - top);
      sum = sum * f + exp2f(sl - top);
    }
    return f / sum * sigmoid_gate(p.x, tok, head);
  }
}

// E4M3 pages: four waves per SIMD at least, or the compiler keeps the output in
// accumulation registers and copies it out and back for every rescale.
template <int D, int NW, int SRC, bool WIDE, int PARTS = 1>  // WIDE: groups of 6 to 8
__global__ __launch_bounds__(NW * 64, SRC == PAGES_FP8 ? 4 : 1) void paged_attention_kernel(
    const DecodeArgs p) {
  constexpr int KC = D / 32;           // contraction chunks of K Q^T
  constexpr int DB = D / 16;           // 16-column blocks of the output
  constexpr int ROWS = 2 * PAGE;       // rows of a stage (a pair of pages)
  constexpr int ES = SRC == PAGES_FP8 ? 1 : 2;
  constexpr int STAGE = ROWS * D * ES;  // shorts: K rows, then V rows
  static_assert(SRC != PAGES_FP8 || D == 128, "E4M3 rows are 8 chunks");
  // elements per lane and load, loads per stage and tensor
  constexpr int EPL = SRC == PAGES_FP8 ? 16 : 8;
  constexpr int LPR = D / EPL;  // lanes per row
  constexpr int RPI = 64 / LPR;
  constexpr int NI = ROWS / RPI;

  const int kvh = blockIdx.x, s = blockIdx.y, split = blockIdx.z;
  const int ctx = p.ctx_lens[s];
  const Range rg = page_range(ctx, p.window, p.x.chunk, p.n_splits, min(NW, WAVES));
  const int tok = token_of(p, s);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // waves with work: the others end here (and are not waited for at the barrier)
  const int nw = NW > WAVES && rg.per < deep_pairs(SRC) ? WAVES : NW;
  if (split >= rg.splits || tok < 0 || wave >= nw) return;
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, g = lane >> 4;
  const int G = p.group;
  const int part = col / G;  // of the weights: high, middle, low
  const bool used = part < (WIDE ? 2 : 3);
  const float past_hi = part > 0 ? 1.f : 0.f, past_mid = part > 1 ? 1.f : 0.f;

  __shared__ __attribute__((aligned(16))) short lds[NW][STAGE];
  static_assert(STAGE * 2 >= 8 * (D + 4) * 4 + 64, "merge area");

  bf16x8_t qf[PARTS][KC];
  {
    const long at = (long)tok * p.sq + (long)(kvh * G + col % G) * D + g * 8;
    if constexpr (PARTS == 1) {
      const short* qp = reinterpret_cast<const short*>(p.q) + at;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        short8_t x = *reinterpret_cast<const short8_t*>(qp + c * 32);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = used ? x[j] : 0;
        qf[0][c] = __builtin_bit_cast(bf16x8_t, x);
      }
    } else {
      const float* qp = reinterpret_cast<const float*>(p.q) + at;
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 8; j += 4) {
          const f32x4_t x = *reinterpret_cast<const f32x4_t*>(qp + c * 32 + j);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const Split3 w(used ? x[e] : 0.f);
            qf[0][c][j + e] = w.hi;
            qf[1][c][j + e] = w.mid;
            qf[2][c][j + e] = w.lo;
          }
        }
    }
  }

  const int* bt = p.block_tables + (long)s * p.max_blocks;
  const int lrow = lane / LPR, lchunk = lane % LPR;
  struct Pages {
    int a, b;
  };
  // page ids of pair n (past the end: the last page again, as its rows are)
  auto pages_of = [&](int n) {
    const int a = min(rg.first + 2 * n, rg.last), b = min(a + 1, rg.last);
    return Pages{bt[a], bt[b]};
  };
  // where this lane's bytes of load i come from; rows past the context repeat
  // its last one (their weights are 0, their values finite)
  auto src = [&](const void* cache, long stride, int n, Pages pg, int i, int chunk) {
    const bool second = i >= NI / 2;
    const int number = min(rg.first + 2 * n + (second ? 1 : 0), rg.last);
    const int row = min((i % (NI / 2)) * RPI + lrow, ctx - 1 - number * PAGE);
    const long st = PARTS == 1 ? D : stride;  // bf16 queries: whole rows
    return reinterpret_cast<const char*>(cache) +
           ((long)(second ? pg.b : pg.a) * p.Hkv + kvh) * PAGE * st * ES +
           (row * (int)st + chunk * EPL) * ES;
  };
  uint4 raw[2 * NI];
  auto load = [&](int n) {
    const Pages pg = pages_of(n);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      raw[2 * i] = load16_nt(src(p.k_cache, p.sk, n, pg, i, lchunk));
      raw[2 * i + 1] = load16_nt(src(p.v_cache, p.sv, n, pg, i, lchunk));
    }
  };
  auto commit = [&]() {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = i * RPI + lrow;
#pragma unroll
      for (int kv = 0; kv < 2; ++kv) {
        char* row = reinterpret_cast<char*>(lds[wave]) + (kv * ROWS + r) * D * ES;
        const int sw = SRC == PAGES_FP8 ? (r >> 1) & 7 : kv ? v_swz<D>(r) : k_swz<D>(r);
        *reinterpret_cast<uint4*>(row + (lchunk ^ sw) * 16) = raw[2 * i + kv];
      }
    }
  };

  // Operand addresses inside a stage (bytes). E4M3 rows stay one byte an element and are
  // widened on the way to the product.
  int kaddr[KC];
#pragma unroll
  for (int c = 0; c < KC; ++c)
    kaddr[c] = SRC == PAGES_FP8
                   ? col * D + ((2 * c + (g >> 1)) ^ (col >> 1)) * 16 + (g & 1) * 8
                   : (col * D + ((4 * c + g) ^ k_swz<D>(col)) * 8) * 2;
  // Transposing load: lane i of 16 brings key i/4, columns 4 (i%4) .. + 3 and
  // receives column i of its four keys; of E4M3 key i/2, columns 8 (i%2) .. + 7 and
  // column i of eight keys, the fragment's of both pages.
  const int vrow = SRC == PAGES_FP8 ? (col >> 3) * PAGE + g * 4 + ((col >> 1) & 3)
                                    : g * 4 + (col >> 2);
  int vaddr[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
    vaddr[b] = SRC == PAGES_FP8
                   ? (ROWS + vrow) * D + (b ^ ((vrow >> 1) & 7)) * 16 + (col & 1) * 8
                   : (ROWS * D + vrow * D + ((2 * b + ((col & 3) >> 1)) ^ v_swz<D>(vrow)) * 8 +
                      (col & 1) * 4) * 2;
  auto widen = [](uint2 x) {  // eight E4M3 bytes, exactly
    uint4 o;
    o.x = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x.x, 1.0f, false));
    o.y = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x.x, 1.0f, true));
    o.z = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x.y, 1.0f, false));
    o.w = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x.y, 1.0f, true));
    return __builtin_bit_cast(bf16x8_t, o);
  };

  float c2 = p.scale * LOG2E;
  const bool flip = c2 < 0.f;
  c2 = fabsf(c2);
  const int key_lo = low_of(ctx - 1, p.window, p.x.chunk);  // first visible key
  float m = NO_MAX, l = 0.f;
  f32x4_t o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) o[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  auto compute = [&](int n, const char* st) {
    f32x4_t sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      f32x4_t rest = sc[h];  // the products with the query's lower parts
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const char* from = st + h * PAGE * D * ES + kaddr[c];
        bf16x8_t a;
        if constexpr (SRC == PAGES_FP8) a = widen(*reinterpret_cast<const uint2*>(from));
        else a = *reinterpret_cast<const bf16x8_t*>(from);
        if constexpr (PARTS == 3) {
          rest = mfma16x16x32(a, qf[PARTS - 1][c], rest);
          rest = mfma16x16x32(a, qf[PARTS - 2][c], rest);
        }
        sc[h] = mfma16x16x32(a, qf[0][c], sc[h]);
      }
      if constexpr (PARTS == 3) sc[h] += rest;
    }
    if (flip) {
      sc[0] = -sc[0];
      sc[1] = -sc[1];
    }
    const int key0 = (rg.first + 2 * n) * PAGE;
    if (key0 + ROWS > ctx || key0 < key_lo) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = key0 + h * PAGE + g * 4 + r;
          sc[h][r] = key < ctx && key >= key_lo ? sc[h][r] : MASKED;
        }
    }
    float mx = fmaxf(fmaxf(fmaxf(sc[0][0], sc[0][1]), fmaxf(sc[0][2], sc[0][3])),
                     fmaxf(fmaxf(sc[1][0], sc[1][1]), fmaxf(sc[1][2], sc[1][3])));
    mx = column_max(mx);
    if (__any(mx > m)) {
      const float mn = fmaxf(m, mx);
      const float f = __builtin_amdgcn_exp2f((m - mn) * c2);
      m = mn;
      l *= f;
#pragma unroll
      for (int b = 0; b < DB; ++b) o[b] *= f;
    }
    const float mc = m * c2;
    bf16x8_t pf, pl;
    if constexpr (WIDE || SRC == PAGES_FP8) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float w = __builtin_amdgcn_exp2f(sc[h][r] * c2 - mc);
          l += w;
          const Split3 w3(w);
          if constexpr (WIDE) {
            pf[h * 4 + r] = part == 0 ? w3.hi : w3.mid;
            pl[h * 4 + r] = part == 0 ? w3.lo : (__bf16)0.f;
          } else {
            pf[h * 4 + r] = part == 0 ? w3.hi : part == 1 ? w3.mid : w3.lo;
          }
        }
    } else {
      // a lane's part by two factors of its own, two weights to a conversion: half of
      // what forming all three and choosing takes (weights are 0 to 1 or NaN; for E4M3
      // the factors' registers are spilled, and scratch costs 1.3 us a launch)
      unsigned int u[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = __builtin_amdgcn_exp2f(sc[i >> 1][(i & 1) * 2] * c2 - mc);
        const float y = __builtin_amdgcn_exp2f(sc[i >> 1][(i & 1) * 2 + 1] * c2 - mc);
        l += x;
        l += y;
        const Rounded2 hi(x, y);
        const float x1 = __builtin_fmaf(-past_hi, hi.first(), x);
        const float y1 = __builtin_fmaf(-past_hi, hi.second(), y);
        const Rounded2 mid(x1, y1);
        u[i] = Rounded2(__builtin_fmaf(-past_mid, mid.first(), x1),
                        __builtin_fmaf(-past_mid, mid.second(), y1)).bits;
      }
      pf = __builtin_bit_cast(bf16x8_t, uint4{u[0], u[1], u[2], u[3]});
    }
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      union {
        s16x4_t h[2];
        bf16x8_t v;
      } a;
      const char* a0 = st + vaddr[b];
      if constexpr (SRC == PAGES_FP8) {
        typedef int i2_t __attribute__((ext_vector_type(2)));
        typedef __attribute__((address_space(3))) i2_t lds2_t;
        a.v = widen(__builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds2_t*)a0)));
      } else {
        typedef __attribute__((address_space(3))) s16x4_t lds4_t;
        a.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)a0);
        a.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)(a0 + PAGE * D * 2));
      }
      o[b] = mfma16x16x32(a.v, pf, o[b]);
      if constexpr (WIDE) o[b] = mfma16x16x32(a.v, pl, o[b]);
    }
  };

  const int n_lo = split * rg.per + wave;
  const int n_hi = min((split + 1) * rg.per, rg.pairs);
  if (n_lo < n_hi) load(n_lo);
  // the next pair's loads are under way while this one is multiplied
  for (int n = n_lo; n < n_hi; n += nw) {
    commit();
    if (n + nw < n_hi) load(n + nw);
    compute(n, reinterpret_cast<const char*>(lds[wave]));
  }

  // ---- merge: the parts of the weights, then the waves ----
  l = column_sum(l);
  float* mo = reinterpret_cast<float*>(lds[wave]);  // [8][D + 4], then m and l
  float* mm = mo + 8 * (D + 4);
#pragma unroll
  for (int b = 0; b < DB; ++b) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = o[b][r] + __shfl(o[b][r], lane + G, 64);
      if constexpr (!WIDE) x += __shfl(o[b][r], lane + 2 * G, 64);
      o[b][r] = x;
    }
    if (col < G)
      *reinterpret_cast<f32x4_t*>(mo + col * (D + 4) + b * 16 + g * 4) = o[b];
  }
  if (lane < G) {
    mm[lane] = m;
    mm[8 + lane] = l;
  }
  __syncthreads();
  constexpr int WF = STAGE / 2;  // floats between the waves' areas
  const float* all = reinterpret_cast<const float*>(lds);
  for (int i = threadIdx.x; i < G * (D / 4); i += nw * 64) {
    const int h = i / (D / 4), d = i % (D / 4) * 4;
    float top = NO_MAX;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (w < nw) top = fmaxf(top, all[w * WF + 8 * (D + 4) + h]);
    float sum = 0.f;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      if (w >= nw) continue;
      const float* a = all + w * WF;
      const float f = __builtin_amdgcn_exp2f((a[8 * (D + 4) + h] - top) * c2);
      sum += f * a[8 * (D + 4) + 8 + h];
      acc += f * *reinterpret_cast<const f32x4_t*>(a + h * (D + 4) + d);
    }
    const int head = kvh * G + h;
    if (rg.splits == 1) {
      const float f = final_factor<PARTS>(p, tok, head, top * c2, sum);
      store4(p.out, ((long)tok * p.H + head) * D + d, acc * f,
             PARTS == 1 ? 0 : p.x.out_f32);
    } else {
      const long at = ((long)s * p.H + head) * p.n_splits + split;
      *reinterpret_cast<f32x4_t*>(p.part_out + at * D + d) = acc;
      if (d == 0) {
        p.part_ml[at * 2] = top * c2;
        p.part_ml[at * 2 + 1] = sum;
      }
    }
  }
}

// Combine split-context partials: one wave per (seq, head); a lane owns D/64
// columns across all splits. Sequences that one split covers are done.
template <int D, int NW, int PARTS = 1>
__global__ __launch_bounds__(256) void paged_attention_reduce_kernel(
    const DecodeArgs p, long total) {
  constexpr int ACC = D / 64;
  const long sh = blockIdx.x * 4L + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (sh >= total) return;
  const int s = sh / p.H;
  const Range rg = page_range(p.ctx_lens[s], p.window, p.x.chunk, p.n_splits, min(NW, WAVES));
  const int tok = token_of(p, s);
  if (rg.splits == 1 || tok < 0) return;
  const float* ml = p.part_ml + sh * p.n_splits * 2;
  float m = NO_MAX * 1e6f;
  for (int sp = lane; sp < rg.splits; sp += 64) m = fmaxf(m, ml[sp * 2]);
  m = wave_reduce_max(m);
  float l = 0.f, acc[ACC];
#pragma unroll
  for (int a = 0; a < ACC; ++a) acc[a] = 0.f;
#pragma unroll 4
  for (int sp = 0; sp < rg.splits; ++sp) {
    const float w = __builtin_amdgcn_exp2f(ml[sp * 2] - m);
    l += w * ml[sp * 2 + 1];
    const float* po = p.part_out + (sh * p.n_splits + sp) * D + lane * ACC;
#pragma unroll
    for (int a = 0; a < ACC; ++a) acc[a] += w * po[a];
  }
  const float f = final_factor<PARTS>(p, tok, sh % p.H, m, l);
  const long at = ((long)tok * p.H + sh % p.H) * D + lane * ACC;
#pragma unroll
  for (int a = 0; a < ACC; ++a) {
    if (PARTS == 3 && p.x.out_f32) reinterpret_cast<float*>(p.out)[at + a] = acc[a] * f;
    else reinterpret_cast<short*>(p.out)[at + a] = float_to_bf16_bits(acc[a] * f);
  }
}

// Two waves per block: 32 KB of LDS, four blocks per compute unit, so one
// block's first loads run under the others' last ones. Four from UNSPLIT_BLOCKS to
// FULL_BLOCKS blocks without splits, and of E4M3 pages.
//
// One wave where a table holds a page pair or two per wave (four of E4M3) and
// the blocks are more than the chip takes at once: the second wave has little or
// nothing to do there and its LDS keeps other blocks out (us, 2 waves / 1: 1000
// of 16 tokens, 32 heads 136 / 82, E4M3 130 / 72, of 32 E4M3 137 / 78; 512 of 64,
// 16 heads 58 / 52; 256 of 16, 32 / 8 heads 16 / 12; level at 1024 blocks). Above,
// the longest sequence's block takes its time (400 +- 60% of 4096 blocks 4% to
// 10% slower).
constexpr long ONE_WAVE_BLOCKS = 2048;

template <int D, int SRC, int PARTS, int NW>
void launch_decode_waves(const DecodeArgs& p, int num_seqs, hipStream_t stream) {
  const dim3 grid(p.Hkv, num_seqs, p.n_splits);
  if (3 * p.group <= 16)
    hipLaunchKernelGGL((paged_attention_kernel<D, NW, SRC, false, PARTS>), grid,
                       dim3(NW * 64), 0, stream, p);
  else
    hipLaunchKernelGGL((paged_attention_kernel<D, NW, SRC, true, PARTS>), grid,
                       dim3(NW * 64), 0, stream, p);
}

// E4M3 pages: four waves, two of which end at once where a split has few pairs. Its
// stages are half as large, so that four take the LDS of two, and long contexts among
// short ones end sooner (us, 2 / 4 waves: 96 of 3000 +- 60% 114.2 / 109.3, 192 of 1500
// 101.8 / 95.4, 250 of 1000 +- 60% 102.6 / 97.5, of 150 20.3 / 22.0; before, with stages
// widened in LDS, 119, 113, 104 and 22.3). Behind where contexts are about as long as
// those from which on all four work (before / now 96 / 128 of 400 +- 60 % 21.3 / 23.3, 24.8
// / 28.3; a higher line moves that to longer ones and gives up 96 of 100 with one of 640,
// 16.9 / 12.6). Not past 4096 blocks (1000 of 16 tokens 23.5 / 35.2) nor in many splits,
// which are short (one of 2000 8.6 / 8.9).
constexpr long MOST_DEEP_BLOCKS = 4096;

// bf16 pages stay with two where splits leave none: four are ahead on long contexts, but
// two of them have nothing to do on short ones, and their LDS keeps other blocks out. Which
// it is only the device knows in a captured step, whose tables are as wide as the longest
// allowed (us, 2 / 4 waves, 8 KV heads: 256 of 2048 +- 60% 350 / 339, of 400 74 / 71, of 200
// 40 / 41, of 100 23 / 28, of 30 13 / 19). Half the LDS, values over the keys once these are
// read, lets more blocks in than memory takes well (64 of 1000 50 -> 57).

// Blocks from which on short contexts have no splits, and none.
constexpr long UNSPLIT_BLOCKS = 192, FULL_BLOCKS = 512;

template <int D, int SRC, int PARTS = 1>
hipError_t launch_decode(const DecodeArgs& p, int num_seqs, hipStream_t stream) {
  const bool few = p.max_blocks <= (SRC == PAGES_FP8 ? 8 : 4);
  const long blocks = (long)num_seqs * p.Hkv;
  if (p.n_splits == 1 && blocks >= UNSPLIT_BLOCKS && blocks < FULL_BLOCKS) {
    launch_decode_waves<D, SRC, PARTS, 2 * WAVES>(p, num_seqs, stream);
  } else if (few && p.n_splits == 1 && blocks >= ONE_WAVE_BLOCKS) {
    launch_decode_waves<D, SRC, PARTS, 1>(p, num_seqs, stream);
  } else {
    if constexpr (SRC == PAGES_FP8) {
      if (p.n_splits <= 2 && blocks < MOST_DEEP_BLOCKS)
        launch_decode_waves<D, SRC, PARTS, 2 * WAVES>(p, num_seqs, stream);
      else
        launch_decode_waves<D, SRC, PARTS, WAVES>(p, num_seqs, stream);
    } else {
      launch_decode_waves<D, SRC, PARTS, WAVES>(p, num_seqs, stream);
    }
  }
  HIP_CHECK_KERNEL();
  if (p.n_splits > 1) {
    const long sh = (long)num_seqs * p.H;
    hipLaunchKernelGGL((paged_attention_reduce_kernel<D, WAVES, PARTS>),
                       dim3((unsigned)((sh + 3) / 4)), dim3(256), 0, stream, p, sh);
    HIP_CHECK_KERNEL();
  }
  return hipSuccess;
}

// Context splits for a launch over num_seqs x num_kv_heads; `light`: pages of 2 KB (E4M3,
// heads of 64), whose blocks take half the LDS. None from FULL_BLOCKS blocks on (8 KV
// heads, us: 64 sequences of 1500 61.5 unsplit, 65 with 2 splits, 69 with 4).
//
// Below, 512 to 960 blocks (light: 640 to 1024), as even a number on each unit as that
// allows (us, about 640 blocks / so: 8 of 1500 16.9 / 15.0, of 4000 29.8 / 25.9, 16 of 900
// 19.0 / 16.9, 40 of 2500 83.5 / 78.1, E4M3 49.2 / 44.8); of counts as even as each other the
// larger up to 640 blocks, since a long context among short ones is what the launch waits
// for (32 of 3000 76.9 / 77.9, but 24 of 100 and one of 7000, 25 in all, 44.6 / 36.2). At most
// 32 (one of 7000: 14 us with 32, 16 with 16). A sequence uses as many of them as it has page
// pairs for every wave.
//
// Tables of few pages have none from UNSPLIT_BLOCKS on: blocks of four waves spare the launch
// that merges (us, split / not: 24 of 100 9.2 / 6.9, of 400 14.2 / 11.8, 32 of 1300 38.4 /
// 37.2, 63 of 1000 53.2 / 50.4, E4M3 33.1 / 28.4; fp32 queries, 4 KV heads, 64 of 200 14.2 /
// 11.2, of 1000 33.7 / 30.0). How few is what one long context among short ones allows: 40
// pages up to 255 blocks (others of 100: 24 with one of 640 11.3 / 11.1, of 1500 14.4 / 18.6,
// of 2000 16.3 / 22.8), 128 at one block a unit and from 384 on (32 with one of 1500 22.9 /
// 18.9, 48 22.1 / 19.3), 40 again between, one on some units and two on the others (40
// of 1200 41 / 42); light pages 16 up to there (24 of 900 E4M3 15.6 / 17.3, heads of 64 12.4 /
// 13.2). The width of the table stands for the longest context: a captured step's is the
// longest that the model allows, so the models of more than 2048 tokens keep their splits
// there (24 of 400 15.0 with 512 pages a row, 12.4 with as many as it needs).
inline int decode_splits(int num_seqs, int num_kv_heads, int max_blocks, bool light) {
  const long base = (long)num_seqs * num_kv_heads;
  if (base <= 0 || base >= FULL_BLOCKS) return 1;
  const int short_pages = base >= 384 ? 128
                          : light     ? 16
                          : base == 256 ? 128
                                        : 40;
  if (base >= UNSPLIT_BLOCKS && max_blocks <= short_pages) return 1;
  const long least = light ? 640 : 512, target = light ? 1024 : 960;
  long n = (least + base - 1) / base;
  // blocks of the busiest unit, each with 1 / t of the context
  auto rounds = [&](long t) { return (base * t + 255) / 256; };
  const long even = (640 + base - 1) / base;  // up to here the larger of two that tie
  for (long t = n + 1; t * base <= target; ++t)
    if (rounds(t) * n < rounds(n) * t + (t <= even)) n = t;
  const long most = ((long)max_blocks + 2 * WAVES - 1) / (2 * WAVES);
  if (n > most) n = most;
  if (n > 32) n = 32;
  return n < 1 ? 1 : (int)n;
}

}  // namespace mfma_attn
}  // namespace
