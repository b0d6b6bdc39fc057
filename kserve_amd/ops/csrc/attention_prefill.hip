// Flash-style prefill attention (bf16, GQA, varlen) on MFMA: rows of the
// current batch (flash_prefill_varlen) or pages of the KV cache
// (context_prefill_varlen: chunked prefill, prefix reuse, draft verification).
//
// The tiles are transposed: S^T = K Q^T puts one query per lane column of
// v_mfma_f32_32x32x16_bf16, so the running maximum, sum and rescale factor are
// per-lane scalars, and the 16 score registers of a lane are already the B
// operand of O^T += V^T P^T: the contraction runs over keys in the
// accumulator's own order (lane half h, element j -> key 4h + j, then
// 8 + 4h + j of a 16-key chunk), and V is read from its row-major LDS tile in
// that order by the transposing LDS loads (ds_read_b64_tr_b16). The weights
// never leave registers.
//
// A block is 4 waves of 32 queries and shares double-buffered tiles of 64 keys
// that the LDS-direct loads fill while the other buffer is computed on; the
// XOR swizzles below are on the source side of those loads. With several query
// heads per KV head the waves take up to four heads of one group over the same
// queries (equal causal ranges, and a K/V tile is fetched once for the group);
// otherwise consecutive queries of one head.
//
// What bounds it: per 64 keys and 32 queries a wave issues 32 MFMAs (1024
// cycles of its matrix core), reads 32 KB of LDS operands (a quarter of the
// LDS bandwidth for the same time, times four waves) and has 32 exponentials
// and about 130 further vector instructions per lane; two waves per SIMD
// overlap the three. Measured (32 query and 8 KV heads of 128, causal; the
// 16x16x32 kernel with one head per block, V transposed by 2-byte LDS stores and
// a barrier on each side of the staging, before this one): 1 x 8191 tokens
// 2497 -> 652 us (220 -> 843 TFLOP/s), 8 x 2048 1280 -> 387 us, 32 x 512
// 413 -> 149 us; 2 x 1000 queries over 13000 paged keys 2441 -> 509 us (E4M3
// pages 2596 -> 625); 64 x 128, 12 heads of 64, bidirectional 28 -> 13 us.
//
// Replaces the vLLM flash prefill the reference delegates to
// (SURVEY.md §2.7 row 1). Numerics oracles: ops/torch_ref.flash_prefill_varlen
// and context_attention_varlen.
#include "common.h"
#include "mfma_layouts.h"

namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));

constexpr int KT = 64;      // keys per tile
constexpr int NWAVES = 4;
constexpr int QW = 32;      // queries per wave
constexpr float MASKED = -3e38f;
constexpr float NO_MAX = -1e30f;  // above MASKED: an all-masked tile adds 0

// where K and V rows come from
enum Src {
  ROWS_DMA,   // flat rows, 16-byte aligned: loaded straight into LDS
  ROWS_REG,   // flat rows at any alignment: through registers
  PAGES_DMA,  // bf16 pages of 16 tokens
  PAGES_REG,  // bf16 pages at any alignment
  PAGES_FP8,  // E4M3 pages, widened to bf16 on the way
};

// 16-byte chunk that chunk c of row r sits at. K fragments: 16 consecutive
// rows at one chunk must hit different banks; V fragments: 4 consecutive rows
// of 32 bytes each (a pair of chunks stays a pair).
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

struct PrefillArgs {
  short* out;         // [T, Hq, D]
  const short* q;     // [T, Hq, D], row stride sq
  const void* k;      // [T, Hkv, D] rows (stride sk) or pages [NB, Hkv, 16, D]
  const void* v;
  const int* cu_q;          // [S+1]
  const int* ctx_lens;      // [S] keys of a sequence (pages)
  const int* block_tables;  // [S, max_nb] (pages)
  int Hq, Hkv, max_nb;
  int hpb;  // query heads per block: 1, 2 or 4, divides the group
  float scale;
  long sq, sk, sv;
  int window;
};

template <int D, int SRC, bool CAUSAL, bool WIN>
__global__ __launch_bounds__(256, 2) void prefill_attention_kernel(
    const PrefillArgs p) {
  constexpr bool PAGED = SRC >= PAGES_DMA;
  constexpr bool DMA = SRC == ROWS_DMA || SRC == PAGES_DMA;
  constexpr int CPR = D / 8;          // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;       // rows per wave-wide 16-byte load
  constexpr int NI = 16 / RPI;        // such loads per wave and tile (K or V)
  constexpr int TILE = KT * D;
  constexpr int KC = D / 16;          // contraction chunks of Q K^T
  constexpr int DB = D / 32;          // 32-column blocks of the output

  const int seq = blockIdx.z;
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

  // ---- queries: B operands, 8 consecutive columns per lane ----
  bf16x8_t qf[KC];
  {
    const int qrow = min(q0 + (lane & 31), q_len - 1);
    const short* qp = p.q + (long)(q_start + qrow) * p.sq + (long)head * D + half * 8;
#pragma unroll
    for (int c = 0; c < KC; ++c)
      qf[c] = *reinterpret_cast<const bf16x8_t*>(qp + c * 16);
  }

  // ---- key range ----
  const int last_q = min(tile_base + qpb, q_len) - 1;
  const int hi = CAUSAL ? min(len, start_pos + last_q + 1) : len;
  const int lo = WIN ? max(0, start_pos + tile_base - p.window + 1) : 0;
  const int t_lo = lo / KT;
  const int t_hi = (hi + KT - 1) / KT;
  const int pos_lo = start_pos + q0;
  const int pos_hi = start_pos + min(q0 + QW, q_len) - 1;
  const int my_pos = start_pos + q0 + (lane & 31);

  // ---- staging: wave w brings rows 16 w .. 16 w + 15 of a tile (one page);
  // rows past the keys repeat the last one (their weights are 0, their values
  // finite) ----
  const int* bt = PAGED ? p.block_tables + (long)seq * p.max_nb : nullptr;
  const int lrow = lane / CPR, lchunk = lane % CPR;
  auto group_of = [&](int t) { return min(t * KT + wave * 16, len - 1); };
  auto page_of = [&](int t) { return PAGED ? bt[group_of(t) >> 4] : 0; };
  // address of this lane's chunk (c, already unswizzled) of row r of tile t
  auto src = [&](const void* base, long stride, int t, int page, int r, int c) {
    const int g0 = PAGED ? group_of(t) & ~15 : group_of(t);
    const int row = min(r, len - 1 - g0);
    if constexpr (PAGED) {
      constexpr int ES = SRC == PAGES_FP8 ? 1 : 2;
      return reinterpret_cast<const char*>(base) +
             ((long)page * p.Hkv + kvh) * (16 * D * ES) + (row * D + c * 8) * ES;
    } else {
      return reinterpret_cast<const char*>(base) +
             ((long)(q_start + g0) * stride + (long)kvh * D) * 2 +
             (long)row * stride * 2 + c * 16;
    }
  };
  uint2 raw8[SRC == PAGES_FP8 ? 2 * NI : 1];
  short8_t raw16[!DMA && SRC != PAGES_FP8 ? 2 * NI : 1];
  // DMA: fills buffer `buf`; otherwise the rows wait in registers for commit()
  auto stage = [&](int t, int page, int buf) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = i * RPI + lrow;
      const char* ks = src(p.k, p.sk, t, page, r, lchunk ^ k_swz<D>(r));
      const char* vs = src(p.v, p.sv, t, page, r, lchunk ^ v_swz<D>(r));
      if constexpr (DMA) {
        const int at = (wave * 16 + i * RPI) * D;
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const unsigned int*>(ks),
            reinterpret_cast<unsigned int*>(&lds[buf][0][at]), 16, 0, 0);
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const unsigned int*>(vs),
            reinterpret_cast<unsigned int*>(&lds[buf][1][at]), 16, 0, 0);
      } else if constexpr (SRC == PAGES_FP8) {
        raw8[2 * i] = *reinterpret_cast<const uint2*>(ks);
        raw8[2 * i + 1] = *reinterpret_cast<const uint2*>(vs);
      } else {
        raw16[2 * i] = *reinterpret_cast<const short8_t*>(ks);
        raw16[2 * i + 1] = *reinterpret_cast<const short8_t*>(vs);
      }
    }
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

  float c2 = p.scale * 1.44269504088896340736f;
  const bool flip = c2 < 0.f;
  c2 = fabsf(c2);
  float m = NO_MAX, l = 0.f;
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
    __syncthreads();
    if (t + 1 < t_hi) {
      stage(t + 1, page, buf ^ 1);
      if (PAGED && t + 2 < t_hi) page = page_of(t + 2);
    }
    const int t0 = t * KT;
    const bool mine = q0 < q_len && (!CAUSAL || t0 <= pos_hi) &&
                      (!WIN || t0 + KT - 1 > pos_lo - p.window);
    if (mine) {
      const short* kt = lds[buf][0];
      const short* vt = lds[buf][1];
      f32x16_t s[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const bf16x8_t a =
              *reinterpret_cast<const bf16x8_t*>(kt + kb * 32 * D + kaddr[c]);
          s[kb] = mfma32(a, qf[c], s[kb]);
        }
      }
      if (flip) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] = -s[kb];
      }
      // register r of block kb: key 32 kb + (r & 3) + 8 (r / 4) + 4 half
      if (t0 + KT > len || (CAUSAL && t0 + KT - 1 > pos_lo) ||
          (WIN && t0 <= pos_hi - p.window)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = t0 + 32 * kb + (r & 3) + 8 * (r >> 2) + 4 * half;
            const bool ok = key < len && (!CAUSAL || key <= my_pos) &&
                            (!WIN || key > my_pos - p.window);
            s[kb][r] = ok ? s[kb][r] : MASKED;
          }
      }
      float mx = s[0][0];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[kb][r]);
      mx = half_max(mx);
      if (__any(mx > m)) {
        const float mn = fmaxf(m, mx);
        const float f = __builtin_amdgcn_exp2f((m - mn) * c2);
        m = mn;
        l *= f;
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[b][r] *= f;
      }
      const float mc = m * c2;
      bf16x8_t pf[KT / 16];
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float w = __builtin_amdgcn_exp2f(s[kb][r] * c2 - mc);
          sum += w;
          pf[kb * 2 + (r >> 3)][r & 7] = (__bf16)w;
        }
      l += sum;
#pragma unroll
      for (int kc = 0; kc < KT / 16; ++kc)
#pragma unroll
        for (int b = 0; b < DB; ++b) {
          typedef __attribute__((address_space(3))) s16x4_t lds4_t;
          const short* a0 = vt + kc * 16 * D + vaddr[b];
          const s16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)a0);
          const s16x4_t v1 =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4_t*)(a0 + 8 * D));
          union {
            s16x4_t h[2];
            bf16x8_t v;
          } a;
          a.h[0] = v0;
          a.h[1] = v1;
          o[b] = mfma32(a.v, pf[kc], o[b]);
        }
    }
    if (t + 1 < t_hi) commit(buf ^ 1);
  }

  if (q0 >= q_len) return;
  const int qrow = q0 + (lane & 31);
  l = half_sum(l);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (qrow < q_len) {
    short* op = p.out + ((long)(q_start + qrow) * p.Hq + head) * D + half * 4;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        short4_t w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = float_to_bf16_bits(o[b][g * 4 + r] * inv);
        *reinterpret_cast<short4_t*>(op + b * 32 + g * 8) = w;
      }
  }
}

template <int D, int SRC>
hipError_t launch(PrefillArgs p, int num_seqs, int max_q_len, bool causal,
                  hipStream_t stream) {
  const int group = p.Hq / p.Hkv;
  p.hpb = group % 4 == 0 ? 4 : group % 2 == 0 ? 2 : 1;
  const int qpb = NWAVES * QW / p.hpb;
  const int tiles = (max_q_len + qpb - 1) / qpb;
  if (tiles == 0 || num_seqs == 0) return hipSuccess;
  const dim3 grid(p.Hq / p.hpb, tiles, num_seqs);
#define GO(CC, WW)                                                             \
  hipLaunchKernelGGL((prefill_attention_kernel<D, SRC, CC, WW>), grid,         \
                     dim3(256), 0, stream, p)
  const bool win = p.window > 0;
  if constexpr (SRC >= PAGES_DMA) {
    if (win) GO(true, true);
    else GO(true, false);
  } else if (causal) {
    if (win) GO(true, true);
    else GO(true, false);
  } else {
    if (win) GO(false, true);
    else GO(false, false);
  }
#undef GO
  HIP_CHECK_KERNEL();
  return hipSuccess;
}

bool aligned16(const void* a, const void* b) {
  return (((uintptr_t)a | (uintptr_t)b) & 15) == 0;
}

}  // namespace

extern "C" hipError_t ks_context_prefill_varlen(
    void* out, const void* q, const void* k_cache, const void* v_cache,
    const void* block_tables, const void* ctx_lens, const void* cu_seqlens_q,
    int num_seqs, int max_q_len, int Hq, int Hkv, int head_dim, int max_nb,
    float scale, long sq, int fp8_cache, int window, hipStream_t stream) {
  if (head_dim != 128) return hipErrorInvalidValue;
  if (Hq % Hkv != 0) return hipErrorInvalidValue;
  PrefillArgs p{(short*)out, (const short*)q, k_cache, v_cache,
                (const int*)cu_seqlens_q, (const int*)ctx_lens,
                (const int*)block_tables, Hq, Hkv, max_nb, 1, scale, sq, 0, 0,
                window};
  if (fp8_cache) return launch<128, PAGES_FP8>(p, num_seqs, max_q_len, true, stream);
  if (aligned16(k_cache, v_cache))
    return launch<128, PAGES_DMA>(p, num_seqs, max_q_len, true, stream);
  return launch<128, PAGES_REG>(p, num_seqs, max_q_len, true, stream);
}

extern "C" hipError_t ks_flash_prefill_varlen(
    void* out, const void* q, const void* k, const void* v,
    const void* cu_seqlens, int num_seqs, int max_seqlen, int Hq, int Hkv,
    int head_dim, float scale, long sq, long sk, long sv, int causal,
    int window, hipStream_t stream) {
  if (head_dim != 128 && head_dim != 64) return hipErrorInvalidValue;
  if (Hq % Hkv != 0) return hipErrorInvalidValue;
  PrefillArgs p{(short*)out, (const short*)q, k, v, (const int*)cu_seqlens,
                nullptr, nullptr, Hq, Hkv, 0, 1, scale, sq, sk, sv, window};
  // LDS-direct loads move 16 aligned bytes per lane
  const bool dma = aligned16(k, v) && sk % 8 == 0 && sv % 8 == 0;
  if (head_dim == 128) {
    if (dma) return launch<128, ROWS_DMA>(p, num_seqs, max_seqlen, causal, stream);
    return launch<128, ROWS_REG>(p, num_seqs, max_seqlen, causal, stream);
  }
  if (dma) return launch<64, ROWS_DMA>(p, num_seqs, max_seqlen, causal, stream);
  return launch<64, ROWS_REG>(p, num_seqs, max_seqlen, causal, stream);
}
